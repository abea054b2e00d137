"""GPU parity of the short backward's rank-r part (dS on its own, dA and dB side by side: lora_stream.hip, lora_da_direct.hip) through lf_lora_bwd without the dX
product: one row, ragged rows, every rank tiling and ranks inside one, more columns than one round has workgroups of one tile, padded rows that hold
values, both 16-bit types, masks as bits, as bytes, off the 16-byte grid and none; against float32 sums in torch.  Tolerance: 16-bit results of fp32 sums, 1e-2 of
an element and of the result's root mean square, as everywhere here (oracle.lora_ref.check_close)."""

import ctypes

import pytest
import torch

from oracle import lora_ref
from tests.util import kernels_of

pytestmark = pytest.mark.gpu


def _bwd(dy, x, mask, mask_bits, s, b, a, blocks, scales, ps, valid, ds=None):
    """dS (in `ds`, if given), dA_i, dB_i of one packed batch (blocks: 128-row blocks of each segment; one segment: no routing tables)."""
    from lorafusion_amd import _lib as L

    M, N, K, R, n = dy.shape[0], dy.shape[1], x.shape[1], s.shape[1], len(b)
    ranks = [t.shape[1] for t in b]
    if n == 1:
        r, keep = L.single_routing(ranks[0], scales[0], ps[0]), ()
    else:
        table, first = [], 0
        for seg, nb in enumerate(blocks):
            table += [(ranks[seg], min(128, max(0, valid[seg] - 128 * i)), first) for i in range(nb)]
            first += nb
        per = lambda v: torch.tensor([v[seg] for seg, nb in enumerate(blocks) for _ in range(nb)], dtype=torch.float32, device="cuda")
        keep = (torch.tensor(table, dtype=torch.int32, device="cuda"), per(scales), per(ps))
        r = L.multi_routing([nb * 128 for nb in blocks], ranks, *keep, 128)
    ds = torch.full_like(s, 7) if ds is None else ds
    da, db = [torch.full_like(t, 7) for t in a], [torch.full_like(t, 7) for t in b]
    dt = L.dtype_id(dy.dtype) | (L.LF_MASK_BITS if mask_bits else 0)
    nbytes = L.lib().lf_workspace_bytes(L.LF_OP_BWD, M, N, K, R, ctypes.byref(r))
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")

    def call():
        rc = L.lib().lf_lora_bwd(dy.data_ptr(), x.data_ptr(), None, L.ptr(mask), s.data_ptr(), L.ptr_array(a), L.ptr_array(b), None, L.ptr_array(da), L.ptr_array(db),
                                 ds.data_ptr(), ws.data_ptr(), nbytes, M, N, K, R, ctypes.byref(r), dt, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, rc

    _, names = kernels_of(call)
    del keep
    return ds, da, db, names


def _check(got, exp, name):
    ok, rel, excess = lora_ref.check_close(got.float().cpu(), exp.cpu(), rtol=1e-2)
    assert ok, f"{name}: rel {rel:.3e} excess {excess:.3e}"


@pytest.mark.parametrize("tokens,ranks,N,K,p,mask_kind,dtype", [
    ([1], [16], 256, 128, 0.0, "none", torch.bfloat16),                              # one row; the narrowest K and almost the narrowest N
    ([300], [8], 4096, 4096, 0.1, "bits", torch.bfloat16),                           # rank 8 inside 16 columns, ragged rows
    ([257], [32], 640, 8192, 0.2, "bytes", torch.float16),                           # two blocks and a row; more columns in X than in dY
    ([129], [64], 1408, 384, 0.1, "off", torch.bfloat16),                            # the sliced dS; mask bytes off the grid
    ([200], [40], 1024, 1024, 0.1, "bits", torch.float16),                           # rank 40 inside 48 columns
    ([130], [128], 4096, 1152, 0.25, "bits", torch.bfloat16),                        # two tiles per workgroup at least
    ([130, 1, 256, 90], [8, 16, 32, 64], 1152, 2048, 0.1, "bits", torch.bfloat16),   # adapters of different ranks, one row in a segment
    ([100] * 8, [16] * 8, 2048, 1024, 0.1, "bits", torch.bfloat16),                  # 384 tiles for 256 workgroups
    ([64, 128], [24, 16], 512, 512, 0.0, "none", torch.float16)])
def test_against_float32(tokens, ranks, N, K, p, mask_kind, dtype):
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator(device="cuda").manual_seed(sum(tokens) + N)
    rn = lambda *sh, std=1.0: (torch.randn(*sh, generator=g, device="cuda") * std).to(dtype)
    n, R = len(tokens), (max(ranks) + 15) // 16 * 16
    blocks = [(t + 127) // 128 for t in tokens]
    rows = [t if n == 1 else nb * 128 for t, nb in zip(tokens, blocks)]
    M = sum(rows)
    dy, x, s = rn(M, N), rn(M, K), torch.zeros(M, R, device="cuda", dtype=dtype)
    b, a = [rn(N, r, std=0.1) for r in ranks], [rn(r, K, std=0.1) for r in ranks]
    scales = [1.0, 2.0, 0.5, 4.0, 1.0, 3.0, 2.0, 1.5][:n]
    start = [sum(rows[:i]) for i in range(n)]
    for i in range(n):
        s[start[i]:start[i] + tokens[i], :ranks[i]] = rn(tokens[i], ranks[i])
        x[start[i] + tokens[i]:start[i] + rows[i]] = 3.0   # (S and dS are zero there)
        dy[start[i] + tokens[i]:start[i] + rows[i]] = 5.0
    keep = torch.rand(M, K, generator=g, device="cuda") >= p
    mask = None
    if mask_kind == "bits":
        mask = hip_ops.pack_mask(keep)
    elif mask_kind == "bytes":
        mask = keep.to(torch.uint8)
    elif mask_kind == "off":
        flat = torch.zeros(M * K + 16, dtype=torch.uint8, device="cuda")
        mask = flat[1:1 + M * K].view(M, K).copy_(keep)
    ds, da, db, names = _bwd(dy, x, mask, mask_kind == "bits", s, b, a, blocks, scales, [p] * n, tokens)
    assert "reduce_ds_db" not in names and "dys_dyb" not in names, names
    xt = x.float() * (keep if mask is not None else 1.0) / (1 - (p if mask is not None else 0.0))
    for i in range(n):
        rs, real = slice(start[i], start[i] + rows[i]), slice(start[i], start[i] + tokens[i])
        e = scales[i] * (dy[real].float() @ b[i].float())
        _check(ds[real, :ranks[i]], e, f"dS {i}")
        assert not ds[rs, ranks[i]:].any() and not ds[start[i] + tokens[i]:start[i] + rows[i]].any()
        _check(da[i], ds[real, :ranks[i]].float().T @ xt[real], f"dA {i}")
        _check(db[i], scales[i] * (dy[real].float().T @ s[real, :ranks[i]].float()), f"dB {i}")


@pytest.mark.parametrize("over", ["S", "dY", "apart"])
def test_scratch_over_an_input(over):
    """dS_out is the caller's scratch: over S, or over dY of a call without a dX product, the gradients are what they are with a buffer of its own."""
    g = torch.Generator(device="cuda").manual_seed(5)
    rn = lambda *sh: torch.randn(*sh, generator=g, device="cuda").bfloat16()
    dy, x, s, b, a = rn(300, 512), rn(300, 512), rn(300, 16), [rn(512, 16)], [rn(16, 512)]
    dyf, xf, sf = dy.float(), x.float(), s.float()
    ds = {"S": s, "dY": dy.view(-1)[1024:1024 + 300 * 16].view(300, 16), "apart": None}[over]
    ds, da, db, names = _bwd(dy, x, None, True, s, b, a, [3], [2.0], [0.0], [300], ds)
    assert ("dys_dyb" in names) == (over != "apart"), names
    e = 2 * (dyf @ b[0].float())
    _check(ds, e, "dS")
    _check(da[0], ds.float().T @ xf, "dA")
    _check(db[0], 2 * (dyf.T @ sf), "dB")


def test_long_segments_keep_the_two_passes():
    """One workgroup would walk the 64 blocks of 8192 rows alone: dys_dyb and da in two stages are ahead there."""
    M, N, K = 8192, 1024, 1024
    t = lambda *sh: torch.randn(*sh, device="cuda", dtype=torch.bfloat16)
    *_, names = _bwd(t(M, N), t(M, K), None, True, t(M, 16), [t(N, 16)], [t(16, K)], [64], [1.0], [0.0], [M])
    assert "dys_dyb" in names, names


@pytest.mark.parametrize("M,masked,short", [(300, True, True), (300, False, True), (1500, True, False), (2048, True, False), (2048, False, False)])
def test_either_side_of_the_line(M, masked, short):
    """4096 x 4096 at rank 16: the short way to about 1000 rows of one segment with keep bits; at 2048 the two passes are ahead with a mask (28.0 against 31.0 us) and without."""
    t = lambda *sh: torch.randn(*sh, device="cuda", dtype=torch.bfloat16)
    mask = torch.randint(0, 256, (M, 512), device="cuda", dtype=torch.uint8) if masked else None
    *_, names = _bwd(t(M, 4096), t(M, 4096), mask, True, t(M, 16), [t(4096, 16)], [t(16, 4096)], [(M + 127) // 128], [2.0], [0.1 if masked else 0.0], [M])
    assert ("dys_dyb" not in names) == short, names


def test_segment_without_rows():
    """The last adapter has no row blocks in this batch: its gradients are sums of nothing, in both halves of the launch, and the other's are not touched."""
    g = torch.Generator(device="cuda").manual_seed(11)
    rn = lambda *sh: torch.randn(*sh, generator=g, device="cuda").bfloat16()
    M, N, K = 256, 384, 640
    dy, x, s, b, a = rn(M, N), rn(M, K), rn(M, 16), [rn(N, 16), rn(N, 8)], [rn(16, K), rn(8, K)]
    s[200:] = 0
    ds, da, db, names = _bwd(dy, x, None, True, s, b, a, [2, 0], [2.0, 1.0], [0.0, 0.0], [200, 0])
    assert "dys_dyb" not in names, names
    assert not da[1].any() and not db[1].any()
    _check(ds[:200], 2 * (dy[:200].float() @ b[0].float()), "dS")
    _check(da[0], ds[:200].float().T @ x[:200].float(), "dA")
    _check(db[0], 2 * (dy[:200].float().T @ s[:200].float()), "dB")
