"""Which NF4 weight a backward node reads: the one that codes and quant state name when the backward runs, not the one of the
forward.  On the CPU, with a stand-in for ``lf_nf4_lora_bwd`` that writes down what it is handed; in a process of its own, whose
symbols the stand-in may come before."""

import os
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STAND_IN = r"""
#include "lorafusion_hip.h"
extern "C" {
int calls; lf_nf4_weight seen;
int lf_nf4_lora_bwd(const void*, const void*, const lf_nf4_weight* W, const uint8_t*, const void*, const void* const*, const void* const*, void*,
                    void* const*, void* const*, void*, void*, size_t, int, int, int, int, const lf_routing*, int, void*) {
  calls++, seen = *W;
  return 0;
}
}
"""
SETUP = r"""
import ctypes, gc, sys, weakref
import torch
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from lorafusion_amd import _lib as L
from lorafusion_amd.ops import nf4
L.require_gpu = lambda *a: None
T = lambda *s: torch.randn(*s).bfloat16()
P, q = nf4.quantize_nf4(T(128, 128))
P = P.clone()   # (its own storage, no base)
x, a, b = (t.requires_grad_() for t in (T(4, 128), T(16, 128), T(128, 16)))
routing = L.single_routing(16, 1.0, 0.0)
def attach(tables=()):
    return L.host().attach(T(4, 128), [x], x.detach(), P, nf4.nf4_struct_of(q), [], [a], [b], None, T(4, 16), None, [],
                           ctypes.addressof(routing), list(tables), 16, "Node")
seen = lambda: L.NF4Weight.in_dll(stub, "seen")
"""
CASES = {
    "codes_move": """
y, old = attach(), P.data
P.data = P.data.clone()
y.backward(torch.ones_like(y))
assert seen().packed == P.data_ptr() != old.data_ptr()
""",
    "state_moves": """
y, old = attach(), q.absmax
q.absmax, q.state2.absmax = q.absmax.clone(), q.state2.absmax.clone()
y.backward(torch.ones_like(y))
assert seen().absmax == q.absmax.data_ptr() != old.data_ptr() and seen().absmax2 == q.state2.absmax.data_ptr()
""",
    "hook_unpacks_another_tensor": """
made = []
def unpack(t):
    made.append(t.clone())
    return made[-1]
with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
    y = attach()
y.backward(torch.ones_like(y))
assert seen().packed in [t.data_ptr() for t in made if t.dtype == torch.uint8]
""",
    "a_state_that_no_longer_fits_is_refused": """
y = attach()
q.absmax = q.absmax[:1]
try:
    y.backward(torch.ones_like(y))
except ValueError as e:
    assert "absmax" in str(e)
else:
    raise AssertionError
assert ctypes.c_int.in_dll(stub, "calls").value == 0
""",
    "nothing_of_the_forward_is_held": """
y, old = attach(), weakref.ref(P.untyped_storage())
P.data = P.data.clone()
gc.collect()
assert old() is None
""",
    "a_freed_graph_holds_neither_state_nor_tables": """
t = torch.zeros(8)
y, table, state = attach([t]), weakref.ref(t.untyped_storage()), weakref.ref(q)
del t, q
gc.collect()
assert table() is not None and state() is not None
y.backward(torch.ones_like(y))
gc.collect()
assert table() is None and state() is None and y.grad_fn is not None
""",
}


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    d = tmp_path_factory.mktemp("stand_in")
    (d / "s.cpp").write_text(STAND_IN)
    subprocess.run(["g++", "-shared", "-fPIC", f"-I{ROOT}/include", "-o", d / "s.so", d / "s.cpp"], check=True)
    return str(d / "s.so")


@pytest.mark.parametrize("case", CASES)
def test_weight_of_the_backward(stand_in, case):
    r = subprocess.run([sys.executable, "-c", SETUP + CASES[case], stand_in], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("packed_batch", [False, True])
def test_gradient_after_the_weight_has_moved(packed_batch):
    from lorafusion_amd.ops.multi_lora import fused_linear_multi_lora, prepare_multi_lora_batch_info
    from lorafusion_amd.ops.nf4 import fused_linear_lora_nf4, quantize_nf4

    M, K, N, r = 128, 256, 384, 16
    g = torch.Generator().manual_seed(0)
    t = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    codes, state = quantize_nf4(t(N, K) * 0.02)
    x, dy, a, b = t(M, K).requires_grad_(), t(M, N), t(r, K), t(N, r)
    info = prepare_multi_lora_batch_info([M], [0], [r], [0.0], [2.0], 128)

    def dx(move):
        p = codes.clone()
        if packed_batch:
            y = fused_linear_multi_lora(x[None], p, lora_a_list=[a], lora_b_list=[b], seq_len_list=[M], padded_seq_len_list=[M],
                                        block_to_lookup_table=info.block_to_lookup_table, block_to_dropout_p=info.block_to_dropout_p,
                                        block_to_alpha=info.block_to_alpha, enable_dropout=False, same_dropout_p_value=0.0, max_r=r,
                                        quant_state=state)[0]
        else:
            y = fused_linear_lora_nf4(x, p, state, a, b, 2.0)
        if move:
            old = p.data
            p.data = old.clone()
            old.zero_()   # (still allocated: the place holds something else now)
        return torch.autograd.grad(y, x, dy)[0]

    assert torch.equal(dx(True), dx(False))
