"""GPU parity of the GEMM kernel for outputs of about one round (gemm_mid.hip) at its edges: its 160x128, 128x128, 128x64 and
192x128 tiles are pinned (10 to 13), so that K loops of exactly four steps and a few more, ragged
rows, every kind of rank chunk, both 16-bit types, bias, and waves that lie across two adapters run against the CPU oracle.
Tolerances as in test_gpu_lora_single.py / test_gpu_lora_multi.py."""

import pytest
import torch

from oracle import lora_ref
from tests.test_gpu_lora_multi import _run as run_multi
from tests.test_gpu_lora_single import _run_case as run_single
from tests.util import kernels_of

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[10, 11, 12, 13], ids=["160x128", "128x128", "128x64", "192x128"])
def tile(request):
    from lorafusion_amd import _lib

    assert _lib.lib().lf_set_tile_cfg(request.param) == 0
    yield request.param
    assert _lib.lib().lf_set_tile_cfg(-1) == 0


@pytest.mark.parametrize(
    "M,K,N,r,p,scale",
    [
        (256, 256, 256, 16, 0.0, 2.0),     # four K steps: the first, no loop, the last three
        (1, 384, 256, 16, 0.0, 2.0),       # one row
        (300, 384, 640, 8, 0.2, 4.0),      # ragged rows, rank 8 inside a chunk of 32
        (321, 256, 384, 128, 0.1, 1.0),    # one row in the last tile row; four chunks
        (257, 512, 384, 40, 0.3, 0.5),     # rank 40 inside 48 columns: a second chunk with 8 columns
        (640, 768, 512, 64, 0.1, 3.0),     # a scale that is not a power of two
        (520, 512, 640, 96, 0.1, 1.5),
    ],
)
def test_single(tile, M, K, N, r, p, scale):
    run_single(M, K, N, r, p, scale)


@pytest.mark.parametrize("K,bias", [(256, False), (512, True), (4096, False)])
def test_rows_in_the_upper_half_of_the_last_tile(tile, K, bias):
    """The lower waves of the last tile have no rows and no LoRA term.  With K a multiple of 256 their (empty) skinny operand goes to the stage
    that the upper waves' results leave through."""
    rows = {10: 160, 11: 128, 12: 128, 13: 192}[tile]
    run_single(rows + rows // 2 - 11, K, 512, 16, 0.1, 2.0, bias=bias)


@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("M,N,K", [(300, 256, 256), (224, 384, 4096), (129, 128, 320)])
def test_plain_product(tile, trans_b, M, N, K):
    """No LoRA term in any wave; a product with the identity gives the operand back bit for bit."""
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator().manual_seed(M + K)
    a = torch.randn(M, K, generator=g).bfloat16().cuda()
    b = torch.randn(N, K, generator=g).bfloat16().cuda()
    c = hip_ops.gemm(a, b if trans_b else b.T.contiguous(), trans_b=trans_b, tile_cfg=tile)
    ok, rel, excess = lora_ref.check_close(c.float().cpu(), a.float().cpu() @ b.float().cpu().T, rtol=1e-2)
    assert ok, f"rel {rel:.3e} excess {excess:.3e}"
    eye = torch.eye(256).bfloat16().cuda()
    a = torch.randn(M, 256, generator=g).bfloat16().cuda()
    assert torch.equal(hip_ops.gemm(a, eye, trans_b=trans_b, tile_cfg=tile), a)


def test_single_bias_3d_fp16(tile):
    run_single(512, 512, 640, 16, 0.1, 2.0, bias=True, three_d=True)
    run_single(161, 512, 384, 16, 0.1, 2.0, dtype=torch.float16)
    run_single(768, 256, 512, 32, 0.0, 0.25, dtype=torch.float16, bias=True)


@pytest.mark.parametrize(
    "seq,ranks,p_list,scales",
    [
        ([129, 130, 128], [16, 16, 16], [0.1, 0.1, 0.1], [1.0, 2.0, 4.0]),
        ([200, 50], [16, 64], [0.0, 0.0], [2.0, 0.5]),
        ([1, 127, 128, 129, 5, 300, 77, 64], [16, 32, 16, 8, 64, 16, 16, 32], [0.1] * 8, [1.0, 3.0] * 4),   # 80-row waves across every pair of blocks
        ([150, 260, 40], [96, 40, 128], [0.1, 0.0, 0.25], [0.5, 2.0, 1.0]),
    ],
)
def test_multi(tile, seq, ranks, p_list, scales):
    run_multi(seq, 512, 384, ranks, p_list, scales)


def test_pinned_tile_refuses_what_it_does_not_take(tile):
    """A byte keep-mask and a K loop of fewer than four steps are shape errors when pinned; unpinned, both run on another tile."""
    from lorafusion_amd import _lib
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator().manual_seed(tile)
    dy, w = torch.randn(300, 256, generator=g).bfloat16().cuda(), (torch.randn(256, 384, generator=g) * 0.02).bfloat16().cuda()
    ds, a = (torch.randn(300, 16, generator=g) * 0.1).bfloat16().cuda(), (torch.randn(16, 384, generator=g) * 0.05).bfloat16().cuda()
    mask = (torch.rand(300, 384, generator=g) >= 0.1).cuda()
    with pytest.raises(RuntimeError):
        hip_ops.fused_lora_dyw_dsa(dy, w, ds, a, 0.1, mask)
    with pytest.raises(RuntimeError):
        hip_ops.gemm(dy[:, :192].contiguous(), w[:192], trans_b=False)
    bits = hip_ops.fused_lora_dyw_dsa(dy, w, ds, a, 0.1, hip_ops.pack_mask(mask))
    assert _lib.lib().lf_set_tile_cfg(9) != 0 and _lib.lib().lf_set_tile_cfg(-1) == 0
    bytes_ = hip_ops.fused_lora_dyw_dsa(dy, w, ds, a, 0.1, mask)
    term = torch.where(mask, ds.float() @ a.float() / 0.9, torch.zeros((), device="cuda"))
    exp = (dy.float() @ w.float() + term).cpu()
    for got, name in ((bits, "bits"), (bytes_, "bytes")):
        ok, rel, excess = lora_ref.check_close(got.float().cpu(), exp, rtol=1e-2)
        assert ok, f"{name}: rel {rel:.3e} excess {excess:.3e}"


def test_skinny_operand_at_an_odd_address():
    """B and A as views at a 2-byte offset: the products run on a tile that reads them lane by lane, with them on a dword on this kernel's 128x64."""
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator().manual_seed(3)
    M, K, N, r = 600, 2048, 2048, 16
    x, w = torch.randn(M, K, generator=g).bfloat16().cuda(), (torch.randn(N, K, generator=g) * 0.02).bfloat16().cuda()
    s = (torch.randn(M, r, generator=g) * 0.1).bfloat16().cuda()
    flat = (torch.randn(N * r + 1, generator=g) * 0.05).bfloat16().cuda()
    b, a = flat[1:].view(N, r), flat[1:].view(r, N)
    assert b.data_ptr() % 4 == 2
    for side, kernel in (((b.clone(), a.clone()), "gemm_mid_kernel"), ((b, a), "gemm_lora_kernel")):   # (a copy lies on a dword)
        (y, dx), names = kernels_of(lambda: (hip_ops.fused_lora_xw_sb(x, w, s, side[0], 2.0), hip_ops.fused_lora_dyw_dsa(x, w, s, side[1], 0.0)))
        assert [k for k in ("gemm_mid_kernel", "gemm_lora_kernel") if k in names] == [kernel], names
    for got, exp, name in ((y, x.float() @ w.float().T + 2.0 * s.float() @ b.float().T, "y"), (dx, x.float() @ w.float() + s.float() @ a.float(), "dx")):
        ok, rel, excess = lora_ref.check_close(got.float().cpu(), exp.cpu(), rtol=1e-2)
        assert ok, f"{name}: rel {rel:.3e} excess {excess:.3e}"
