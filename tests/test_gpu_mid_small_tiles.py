"""GPU parity of the 96x64 and 64x64 tiles of the GEMM kernel for outputs of about one round (gemm_mid.hip), whose operands four waves of their own
load: K loops of exactly as many steps as there are stages and a few more, ragged rows, waves of 48 and 32 rows across two adapters, and every kind of rank
chunk, against the CPU oracle.  Tolerances as in test_gpu_lora_single.py / test_gpu_lora_multi.py."""

import re

import pytest
import torch

from oracle import lora_ref
from tests.test_gpu_lora_multi import _run as run_multi
from tests.test_gpu_lora_single import _run_case as run_single
from tests.util import kernels_of

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[14, 15], ids=["96x64", "64x64"])
def tile(request):
    from lorafusion_amd import _lib

    assert _lib.lib().lf_set_tile_cfg(request.param) == 0
    yield request.param
    assert _lib.lib().lf_set_tile_cfg(-1) == 0


@pytest.mark.parametrize(
    "M,K,N,r,p,scale,dtype,bias",
    [
        (1, 256, 256, 16, 0.0, 2.0, torch.bfloat16, False),      # one row, four K steps: no loop between the first and the last three
        (97, 384, 384, 8, 0.2, 4.0, torch.float16, True),        # one row in the last tile row of 96
        (129, 512, 640, 40, 0.3, 0.5, torch.bfloat16, True),     # a second rank chunk with 8 columns
        (300, 4096, 256, 128, 0.1, 1.0, torch.bfloat16, False),  # four chunks
    ],
)
def test_single(tile, M, K, N, r, p, scale, dtype, bias):
    run_single(M, K, N, r, p, scale, dtype=dtype, bias=bias)


def test_multi(tile):
    run_multi([1, 127, 128, 129, 5, 300, 77, 64], 512, 384, [16, 32, 16, 8, 64, 16, 16, 32], [0.1] * 8, [1.0, 3.0] * 4)
    run_multi([150, 260, 40], 256, 384, [96, 40, 128], [0.1, 0.0, 0.25], [0.5, 2.0, 1.0])


def test_short_batches_run_on_them():
    """The plan takes the 96x64 tile for 300 rows over 4096 columns and K (four rows of tiles fill one round).  (Slices of both tiles: test_gpu_split_contraction.py.)"""
    import ctypes

    from lorafusion_amd import _lib
    from lorafusion_amd.ops import hip_ops

    v = (ctypes.c_int * 3)()
    p = [ctypes.cast(ctypes.byref(v, 4 * i), ctypes.POINTER(ctypes.c_int)) for i in range(3)]
    assert _lib.lib().lf_gemm_plan(300, 4096, 4096, 0, *p) == 0 and list(v) == [300, 14, -1]
    x, w = torch.randn(300, 4096).bfloat16().cuda(), torch.randn(4096, 4096).bfloat16().cuda()
    y, names = kernels_of(lambda: hip_ops.gemm(x, w, trans_b=True))
    assert re.findall(r"gemm_mid_kernelI\w+?Lb[01]ELi(\d+)ELi(\d+)E", names) == [("3", "2")] and "ksplit" not in names, names   # (rows and columns / 32)
    ok, rel, excess = lora_ref.check_close(y.float().cpu(), (x.float() @ w.float().T).cpu(), rtol=1e-2)
    assert ok, f"rel {rel:.3e} excess {excess:.3e}"
