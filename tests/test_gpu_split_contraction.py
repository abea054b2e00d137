"""GPU parity of the split contraction: launches with few tiles and a long reduction (left-over rows of a packed
batch, short batches) cut K into slices, keep fp32 partial tiles in the caller's workspace and add them in a
second kernel.  The first two tests run whichever tile the plan picks; slices of each tile by name are at the end.  Checked against the CPU oracle with the tolerance of test_gpu_lora_single.py, and against the same
product through the entry points without a workspace, which never split (fp32 sums in another order: equal to
within one 16-bit step of the result's magnitude).
"""

import re

import pytest
import torch

from oracle import lora_ref
from tests.util import kernels_of, multi_inputs, single_inputs

pytestmark = pytest.mark.gpu

RTOL = 1e-2


def _close(actual, expected, what):
    ok, rel, excess = lora_ref.check_close(actual.detach().float().cpu(), expected, rtol=RTOL)
    assert ok, f"{what}: max|err|/max|e| = {rel:.3e}, worst excess over bound {excess:.3e}"


def _split_bytes(op, M, N, K, R, routing):
    from lorafusion_amd import _lib as L

    return L.lib().lf_workspace_bytes(op, M, N, K, R, routing)


@pytest.mark.parametrize("M,K,N,r,p,dtype,bias,sized", [
    (128, 8192, 256, 16, 0.1, torch.bfloat16, False, "fwd"),     # Y over K = 8192
    (128, 4096, 8192, 16, 0.1, torch.bfloat16, False, "bwd"),    # dX [128, 4096] over N = 8192
    (200, 6144, 2048, 32, 0.1, torch.bfloat16, True, "fwd"),     # ragged rows, bias added by the second kernel
    (64, 8192, 384, 16, 0.0, torch.float16, True, "fwd"),        # fp16, no dropout
    (300, 12288, 512, 64, 0.2, torch.bfloat16, False, "fwd"),    # more than 256 rows, rank 64
    (384, 512, 12288, 16, 0.1, torch.bfloat16, False, None),     # the same for dX (its slices fit the rank-r passes' bytes)
    (1, 8192, 128, 16, 0.1, torch.bfloat16, False, "fwd"),       # a single token
])
def test_single_adapter_split(M, K, N, r, p, dtype, bias, sized):
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops
    from lorafusion_amd.ops.lora_v1 import fused_linear_lora

    routing = L.single_routing(r, 2.0, p)
    R = L.round_rank(r)
    # the size query shows the split where its partial tiles are the largest use of the workspace
    if sized == "fwd":
        assert _split_bytes(L.LF_OP_FWD, M, N, K, R, routing) > _split_bytes(L.LF_OP_XA, M, N, K, R, routing)
    if sized == "bwd":
        rank_r = max(_split_bytes(L.LF_OP_DYS_DYB, M, N, K, R, routing), _split_bytes(L.LF_OP_DA, M, N, K, R, routing))
        assert _split_bytes(L.LF_OP_BWD, M, N, K, R, routing) > rank_r
    d = single_inputs(M, K, N, r, p=p, seed=3, dtype=dtype, bias=bias)
    dev = "cuda"
    x = d["x"].to(dev).requires_grad_(True)
    a = d["a"].to(dev).requires_grad_(True)
    b = d["b"].to(dev).requires_grad_(True)
    w = d["w"].to(dev)
    mask = d["mask"].to(dev) if d["mask"] is not None else None
    bias_t = d["bias"].to(dev) if bias else None
    y = fused_linear_lora(x, w, a, b, 2.0, dropout_p=p, linear_bias=bias_t, dropout_mask=mask)
    y.backward(d["dy"].to(dev))
    torch.cuda.synchronize()
    ye, se = lora_ref.linear_lora_fwd_fp32(d["x"], d["w"], d["a"], d["b"], 2.0, d["mask"], p, d["bias"])
    dxe, dae, dbe, _ = lora_ref.linear_lora_bwd_fp32(d["dy"], d["x"], d["w"], d["a"], d["b"], 2.0, d["mask"], p)
    _close(y, ye, "y")
    _close(x.grad, dxe, "dx")
    _close(a.grad, dae, "da")
    _close(b.grad, dbe, "db")

    # the same forward product through the entry point without a workspace (one launch, no split)
    s, _, _ = hip_ops.fused_dropout_matmul(x.detach(), a.detach(), dropout_p=p, dropout_mask=mask) if p > 0 else \
        hip_ops.fused_dropout_matmul(x.detach(), a.detach(), dropout_p=0.0)
    y1 = hip_ops.fused_lora_xw_sb(x.detach(), w, s, b.detach(), 2.0, bias=bias_t)
    step = float(y1.float().abs().max()) * 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    assert float((y.detach().float() - y1.float()).abs().max()) <= step


def test_left_over_rows_of_a_packed_batch():
    """Two adapters, 256 + 128 padded rows over K = 4096 forward, N = 4096 backward (few enough for one launch of small tiles now; rows behind whole rounds of
    large tiles, in slices: test_left_over_rows_in_slices)."""
    from lorafusion_amd.ops.multi_lora import fused_linear_multi_lora, prepare_multi_lora_batch_info

    seq, ranks, p_list, scales = [250, 100], [16, 32], [0.1, 0.05], [2.0, 0.5]
    K, N = 4096, 4096
    d = multi_inputs(seq, K, N, ranks, p_list, seed=5)
    info = prepare_multi_lora_batch_info(seq, [0, 1], ranks, p_list, scales, 128, output_dtype=torch.float32)
    dev = "cuda"
    x = d["x"].to(dev).requires_grad_(True)
    a_list = [a.to(dev).requires_grad_(True) for a in d["a_list"]]
    b_list = [b.to(dev).requires_grad_(True) for b in d["b_list"]]
    y = fused_linear_multi_lora(
        x.unsqueeze(0), d["w"].to(dev), lora_a_list=a_list, lora_b_list=b_list, seq_len_list=seq,
        padded_seq_len_list=info.padded_seq_len_list, block_to_lookup_table=info.block_to_lookup_table,
        block_to_dropout_p=info.block_to_dropout_p, block_to_alpha=info.block_to_alpha,
        enable_dropout=info.enable_dropout, same_dropout_p_value=info.same_dropout_p_value, max_r=info.max_r,
        dropout_mask=d["mask"].to(dev),
    )
    y.backward(d["dy"].to(dev).unsqueeze(0))
    torch.cuda.synchronize()
    ye, _ = lora_ref.linear_multi_lora_fwd_fp32(d["x"], d["w"], d["a_list"], d["b_list"], seq, d["padded"], scales, p_list,
                                                d["mask"], None)
    dxe, dae, dbe, _ = lora_ref.linear_multi_lora_bwd_fp32(d["dy"], d["x"], d["w"], d["a_list"], d["b_list"], seq,
                                                           d["padded"], scales, p_list, d["mask"])
    _close(y[0], ye, "y")
    _close(x.grad, dxe, "dx")
    for i in range(2):
        _close(a_list[i].grad, dae[i], f"da[{i}]")
        _close(b_list[i].grad, dbe[i], f"db[{i}]")


def _product_kernels(names):
    """(kernel, rows, columns) of every product kernel in a profile's (mangled) names: gemm_mid_kernel<T, NN, rows / 32, columns / 32>, gemm_lora_kernel<T, rows, columns, ...>.  (The
    profiler takes names of bf16 dX products for demangled ones and loses their numbers: the tests below run dX in fp16.)"""
    mid, general = re.findall(r"gemm_mid_kernelI\w+?Lb[01]ELi(\d+)ELi(\d+)E", names), re.findall(r"gemm_lora_kernelI\w+?Li(\d+)ELi(\d+)E", names)
    return {("mid", 32 * int(m), 32 * int(n)) for m, n in mid} | {("general", int(m), int(n)) for m, n in general} | {("persistent", 0, 0) for _ in re.findall("gemm_big_kernel", names)}


# Sizes whose plan is slices of that tile, uneven ones (the last slice is the shortest, every slice but the first starts inside K); ragged rows.
@pytest.mark.parametrize("nn", [False, True], ids=["Y", "dX"])
@pytest.mark.parametrize("tile,M,N,K,r,dtype", [
    (("mid", 64, 64), 21, 128, 12800, 16, torch.bfloat16), (("mid", 96, 64), 65, 3072, 3072, 40, torch.float16), (("mid", 128, 64), 97, 3072, 3072, 16, torch.bfloat16),
    (("mid", 128, 128), 193, 3072, 6144, 64, torch.bfloat16), (("mid", 160, 128), 129, 2560, 10240, 16, torch.float16), (("mid", 192, 128), 161, 2560, 12800, 8, torch.bfloat16)])
def test_slices_of_each_tile(tile, M, N, K, r, dtype, nn):
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    g, dtype = torch.Generator(device="cuda").manual_seed(M + K), torch.float16 if nn else dtype
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).to(dtype)
    R, p = L.round_rank(r), 0.1   # (without a mask a forward of so few rows is one pass over the weight)
    routing, x, w, a, b = L.single_routing(r, 2.0, p), rn(M, K), rn(N, K, std=0.02), rn(r, K, std=K ** -0.5), rn(N, r, std=0.05)
    if not nn:
        bits = hip_ops.pack_mask(torch.rand(M, K, generator=g, device="cuda") >= p)
        (y, s), names = kernels_of(lambda: hip_ops.lora_forward(x, w, [a], [b], routing, R, bits, None))
        exp = x.float() @ w.float().T + 2.0 * s[:, :r].float() @ b.float().T
    else:   # dX [M, N] over K: x in the place of dY, weight [K, N], A [r, N], B [K, r]
        xs, st, keep = rn(M, N), rn(M, R, std=0.1), torch.rand(M, N, generator=g, device="cuda") >= p
        wt, at, bt, bits = w.T.contiguous(), b.T.contiguous(), a.T.contiguous(), hip_ops.pack_mask(keep)
        out, names = kernels_of(lambda: hip_ops.lora_backward(x, xs, wt, [at], [bt], st, routing, R, bits, [r]))
        y, ds = out[0], hip_ops.fused_lora_dys_dyb(x, bt, st, 2.0)[1][:, :r].float()
        exp = x.float() @ wt.float() + torch.where(keep, ds @ at.float() / (1 - p), torch.zeros((), device="cuda"))
    assert _product_kernels(names) == {tile} and "ksplit_reduce_kernel" in names, names
    _close(y, exp.cpu(), "dx" if nn else "y")


@pytest.mark.parametrize("nn", [False, True], ids=["Y", "dX"])
@pytest.mark.parametrize("tile,N,K", [(("mid", 96, 64), 256, 4864), (("mid", 192, 128), 1024, 6912), (("mid", 160, 128), 1536, 3840)])
def test_slices_over_routing_blocks(tile, N, K, nn):
    """Tiles of 96, 160 and 192 rows lie across two adapters; slices of K beside adapters of other ranks and rates."""
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops
    from lorafusion_amd.ops.multi_lora import prepare_multi_lora_batch_info

    seq, ranks, p_list, scales = [130, 380, 500, 200], [16, 8, 32, 16], [0.1, 0.0, 0.2, 0.1], [1.0, 2.0, 0.5, 4.0]   # 2 + 3 + 4 + 2 blocks
    info = prepare_multi_lora_batch_info(seq, list(range(4)), ranks, p_list, scales, 128)
    padded = info.padded_seq_len_list
    routing = hip_ops.MultiRouting(padded, ranks, info.block_to_lookup_table, info.block_to_alpha, info.block_to_dropout_p)
    M, R, start = sum(padded), routing.R, [sum(padded[:i]) for i in range(4)]
    g, dtype = torch.Generator(device="cuda").manual_seed(N + K), torch.float16 if nn else torch.bfloat16
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).to(dtype)
    x, w = rn(M, K), rn(N, K, std=0.02)
    a, b = [rn(r, K, std=K ** -0.5) for r in ranks], [rn(N, r, std=0.05) for r in ranks]
    if not nn:
        (y, s), names = kernels_of(lambda: hip_ops.lora_forward(x, w, a, b, routing.c, R, hip_ops.pack_mask(torch.ones(M, K, dtype=torch.bool, device="cuda")), None))
        exp = x.float() @ w.float().T
        for c, m, r, t, k in zip(start, seq, ranks, b, scales):
            exp[c:c + m] += k * s[c:c + m, :r].float() @ t.float().T
    else:
        xs, s, keep = rn(M, N), torch.zeros(M, R, dtype=dtype, device="cuda"), torch.rand(M, N, generator=g, device="cuda") >= 0.15
        wt, at, bt = w.T.contiguous(), [t.T.contiguous() for t in b], [t.T.contiguous() for t in a]
        for c, m, r in zip(start, seq, ranks):
            s[c:c + m, :r] = rn(m, r)
        out, names = kernels_of(lambda: hip_ops.lora_backward(x, xs, wt, at, bt, s, routing.c, R, hip_ops.pack_mask(keep), ranks))
        y, exp = out[0], x.float() @ wt.float()
        for c, m, r, t, u, k, p in zip(start, seq, ranks, at, bt, scales, p_list):
            term = (k * (x[c:c + m].float() @ u.float())).to(dtype).float() @ t.float() / (1 - p)
            exp[c:c + m] += torch.where(keep[c:c + m], term, torch.zeros((), device="cuda")) if p > 0 else term
    assert _product_kernels(names) == {tile} and "ksplit_reduce_kernel" in names, names
    real = torch.cat([torch.arange(c, c + m) for c, m in zip(start, seq)])
    _close(y[real.cuda()], exp.cpu()[real], "dx" if nn else "y")


def test_left_over_rows_in_slices():
    """4882 rows: 4864 as 256x256 tiles, 18 in five slices of 64x64 tiles, behind them (row0 > 0) and with a rank term of their own rows."""
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    M, N, K, r = 4882, 3200, 3584, 16
    g = torch.Generator(device="cuda").manual_seed(7)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    x, w, a, b = rn(M, K), rn(N, K, std=0.02), rn(r, K, std=K ** -0.5), rn(N, r, std=0.05)
    (y, s), names = kernels_of(lambda: hip_ops.lora_forward(x, w, [a], [b], L.single_routing(r, 2.0, 0.0), L.round_rank(r), None, None))
    assert _product_kernels(names) == {("persistent", 0, 0), ("mid", 64, 64)} and "ksplit_reduce_kernel" in names, names
    exp = x[4800:].float() @ w.float().T + 2.0 * s[4800:, :r].float() @ b.float().T
    _close(y[4800:], exp.cpu(), "y")
