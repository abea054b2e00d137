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
    (1, 128, 8, torch.bfloat16), (65, 1152, 16, torch.float16), (1000, 256, 24, torch.bfloat16),
    (1, 4096, 8, torch.bfloat16), (65, 4224, 16, torch.float16), (1000, 4096, 24, torch.bfloat16),   # (ranks up to 32: sliced from K = 4096, with a mask)
    (3000, 1536, 56, torch.float16), (7040, 1152, 64, torch.bfloat16)])                              # rank 64: sliced, and too short a K for its rows
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
        if mask is not None:
            assert torch.equal(hip_ops._xa(x, mask.cuda(), [a], routing, M, K, R), s), "one byte per element"
    ye, se = lora_ref.linear_lora_fwd_fp32(d["x"], d["w"], d["a"], d["b"], 2.0, mask, p)
    _close(s[:, :r], se, "S")
    _close(y, ye, "Y")
    assert not s[:, r:].any()


@pytest.mark.parametrize("mode", ["given", "drawn"])
@pytest.mark.parametrize("seq,ranks,K", [([1, 129, 64], [64, 8, 40], 512), ([200, 130], [128, 16], 1280), ([70, 1, 300], [16, 8, 24], 4096)])
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


def _xa_entries(x, gu, a_list, routing_c, R):
    """The rank-r entry points that take no workspace, and lf_lora_xa with and without one; each returns S."""
    import ctypes

    from lorafusion_amd import _lib as L

    M, K = x.shape
    lib, st, ap = L.lib(), L.stream_of(x), L.ptr_array(a_list)
    dt = L.dtype_id(x.dtype) | L.LF_MASK_BITS
    nbytes = lib.lf_workspace_bytes(L.LF_OP_XA, M, 0, K, R, routing_c)
    ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device="cuda")

    def call(name, *args):
        s = torch.full((M, R), float("nan"), dtype=x.dtype, device="cuda")
        L.check(getattr(lib, name)(*[s.data_ptr() if v is s_here else v for v in args]), name)
        return s

    s_here = object()
    tail = (M, K, R, routing_c)
    return dict(
        given=lambda size, m=None: call("lf_lora_xa", x.data_ptr(), L.ptr(m), ap, s_here, ws.data_ptr() if size else None, nbytes if size else 0, *tail, dt, st),
        drawn=lambda m: call("lf_lora_xa_seeded", x.data_ptr(), m.data_ptr(), ap, s_here, *tail, ctypes.c_uint64(7), dt, st),
        silu=lambda c, given, m: call("lf_lora_xa_silu_mul", gu.data_ptr(), gu[:, K:].data_ptr(), 2 * K, c.data_ptr(), L.ptr(given), L.ptr(m),
                                      ctypes.c_uint64(7), ap, s_here, *tail, dt, st)), nbytes


def _rank_pass_setup(M, K, ranks, dtype):
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops, norm_act
    from lorafusion_amd.ops.multi_lora import prepare_multi_lora_batch_info

    g = torch.Generator().manual_seed(M + K)
    n, p_list = len(ranks), [0.1, 0.0, 0.3][:len(ranks)]
    keep, p_rows = None, 0.1
    if n == 1:
        routing_c, R = L.single_routing(ranks[0], 1.0, 0.1), L.round_rank(ranks[0])
    else:
        info = prepare_multi_lora_batch_info([100, 128, 3], list(range(n)), ranks, p_list, [1.0] * n, 128, output_dtype=torch.float32)
        keep = hip_ops.MultiRouting(info.padded_seq_len_list, ranks, info.block_to_lookup_table, info.block_to_alpha, info.block_to_dropout_p)
        routing_c, R, p_rows = keep.c, keep.R, np.repeat(np.asarray(p_list, np.float32), 128)
    gu = (torch.randn(M, 2 * K, generator=g) * 1.5).to(dtype).cuda()
    a = [(torch.randn(r, K, generator=g) * K ** -0.5).to(dtype).cuda() for r in ranks]
    c = norm_act.silu_mul_merged(gu)
    xa, nbytes = _xa_entries(c, gu, a, routing_c, R)
    bits = torch.from_numpy(np.packbits(od.keep_mask(M, K, p_rows, 7), axis=1, bitorder="little")).cuda()
    return xa, nbytes, c, bits, (a, keep)


def _without_a_workspace(xa, c, bits):
    """S of the entry points that take no workspace and of lf_lora_xa without one: the same, bit for bit, like the masks they draw."""
    drawn, drawn2 = torch.zeros_like(bits), torch.zeros_like(bits)
    s = xa["given"](False, bits)
    assert torch.isfinite(s).all()
    assert torch.equal(xa["drawn"](drawn), s) and torch.equal(drawn, bits)
    for given, m in ((bits, None), (None, drawn2)):
        x = torch.empty_like(c)
        assert torch.equal(xa["silu"](x, given, m), s) and torch.equal(x, c)
    assert torch.equal(drawn2, bits)
    return s


@pytest.mark.parametrize("M,K,ranks,dtype", [(500, 5120, [128], torch.float16), (2900, 2560, [72], torch.float16), (65, 1152, [128], torch.bfloat16),
                                             (384, 2048, [8, 128, 16], torch.float16)])
def test_high_ranks_without_a_workspace(M, K, ranks, dtype):
    """Above 64 rank columns S is the sliced pass's whether or not the caller gives memory for the slices' sums, bit for bit."""
    xa, nbytes, c, bits, keep = _rank_pass_setup(M, K, ranks, dtype)
    assert nbytes > 0, "several slices"
    assert torch.equal(_without_a_workspace(xa, c, bits), xa["given"](True, bits))
    assert torch.equal(xa["given"](False), xa["given"](True))


@pytest.mark.parametrize("M,K,ranks,dtype", [
    (300, 4096, [16], torch.bfloat16), (1000, 4480, [24], torch.float16), (17, 1920, [64], torch.bfloat16), (65, 2560, [48], torch.float16),
    (2901, 5120, [64], torch.bfloat16), (384, 2048, [8, 64, 16], torch.float16), (384, 4096, [16, 8, 16], torch.bfloat16)])
def test_rank_pass_without_a_workspace(M, K, ranks, dtype):
    """To 64 rank columns the sums are in another order without the memory: one rounding of S apart."""
    xa, nbytes, c, bits, keep = _rank_pass_setup(M, K, ranks, dtype)
    assert nbytes > 0, "the sliced pass, given memory"
    _close(_without_a_workspace(xa, c, bits), xa["given"](True, bits).float().cpu(), "S")
    _close(xa["given"](False), xa["given"](True).float().cpu(), "S, no mask")


@pytest.mark.parametrize("M,K,r", [(300, 4096, 16), (64, 14336, 32)])
def test_rank_pass_without_a_workspace_shares_k(M, K, r):
    """... and takes at most about three times as long (one workgroup that walks all of K: 4 to 8 times)."""
    from lorafusion_amd import _lib as L

    x, a = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(r, K, device="cuda").bfloat16()
    bits = torch.full((M, K // 8), 255, dtype=torch.uint8, device="cuda")
    xa, _ = _xa_entries(x, x, [a], L.single_routing(r, 1.0, 0.1), r)

    def us(f):
        best = float("inf")
        for _ in range(5):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            f()
            t0.record()
            for _ in range(20):
                f()
            t1.record()
            torch.cuda.synchronize()
            best = min(best, t0.elapsed_time(t1) * 50)
        return best

    drawn = bits.clone()
    with_ws, without, seeded = us(lambda: xa["given"](True, bits)), us(lambda: xa["given"](False, bits)), us(lambda: xa["drawn"](drawn))
    print(f"{M} x {K}, rank {r}: {with_ws:.1f} us with a workspace, {without:.1f} without, {seeded:.1f} drawn", flush=True)
    assert without <= 3 * with_ws + 10 and seeded <= 3 * with_ws + 10


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
