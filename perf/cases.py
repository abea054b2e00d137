"""The work a user has this framework do, as cases that can be timed and compared.

A case is a dict of plain values.  ``listed()`` gives the fixed ones, ``draw(rng)`` one more of the same ranges,
``prepare(case, seed)`` what a program holds before the call (tensors, modules, batch tables), ``run(state)`` one pass
through the public entry points, ``work(case)`` the bytes and operations the pass cannot do without and
``tolerance(case)`` how far another correct implementation of the same precision may be off.

Kinds of case:

* ``evaluate``  one adapter, forward only, no dropout (validation, generation): ``fused_linear_lora`` under ``no_grad``
* ``train``     one adapter, forward + backward: ``fused_linear_lora``
* ``packed``    several adapters' segments in one batch, forward + backward: ``fused_linear_multi_lora``
* ``nf4``       one adapter over an NF4 base weight, forward + backward: ``fused_linear_lora_nf4``
* ``dequant``   the NF4 weight alone: ``dequantize_nf4_triton``
* ``norm_act``  RMSNorm and SiLU-multiply, forward + backward: ``rms_norm``, ``silu_mul_merged``
* ``layer``     the linears, norms and activation of a decoder layer over a packed batch, forward + backward, through the
                ``MultiLoRAManager`` and the patched layer's modules (16-bit or NF4 base weights)
"""

from __future__ import annotations

import math
import random

import torch

from lorafusion_amd.ops import multi_lora
from lorafusion_amd.ops.lora_v1 import fused_linear_lora
from lorafusion_amd.ops.multi_lora import fused_linear_multi_lora, prepare_multi_lora_batch_info
from lorafusion_amd.ops.nf4 import dequantize_nf4_triton, fused_linear_lora_nf4, quantize_nf4
from lorafusion_amd.ops.norm_act import rms_norm, silu_mul_merged
from lorafusion_amd.patch.patch_lora import lora_forward, swiglu_lora_forward
from lorafusion_amd.patch.patch_transformers import DecoderLayerLoRAProjections

BLOCK = 128
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # a few sequences generating one token each (or a very short validation batch) through one adapted projection
        dict(name="evaluate_6", kind="evaluate", tokens=6, k=4096, n=4096, rank=16, dtype="bf16", bias=False),
        # validation of one ragged prompt through a wide projection with a bias
        dict(name="evaluate_333", kind="evaluate", tokens=333, k=4096, n=14336, rank=32, dtype="fp16", bias=True),
        # a micro-batch of one ragged sample
        dict(name="train_300", kind="train", tokens=300, k=4096, n=4096, rank=16, p=0.1, dtype="bf16", bias=False, mask="drawn"),
        # the single LoRA linear of the kernel benchmark's smallest row
        dict(name="train_2048", kind="train", tokens=2048, k=4096, n=4096, rank=16, p=0.1, dtype="bf16", bias=False, mask="drawn"),
        # the largest rank, the other 16-bit type, a bias and a keep-mask that the caller supplies
        dict(name="train_rank128", kind="train", tokens=3000, k=5120, n=5120, rank=128, p=0.05, dtype="fp16", bias=True, mask="given"),
        # a short packed batch of adapters of different ranks; ragged segments
        dict(name="packed_1000", kind="packed", tokens=1000, adapters=4, ranks="mixed", k=4096, n=4096, p=0.1, dtype="bf16"),
        # the packed batch of the kernel benchmark: four adapters, 8192 tokens
        dict(name="packed_8192", kind="packed", tokens=8192, adapters=4, ranks="16", k=4096, n=4096, p=0.1, dtype="bf16"),
        # QLoRA: the gate or up projection of an 8B-class layer
        dict(name="nf4_4096", kind="nf4", tokens=4096, k=4096, n=14336, rank=16, p=0.05, dtype="bf16"),
        # loading / merging: the same weight dequantised alone
        dict(name="dequant", kind="dequant", k=4096, n=14336, blocksize=64, nested=True, dtype="bf16"),
        # the streaming kernels either side of the linears, a ragged batch
        dict(name="norm_act_4001", kind="norm_act", tokens=4001, hidden=4096, mlp=14336, train_norm=True, dtype="bf16"),
        # an 8B-class decoder layer over the largest micro-batch of the headline benchmark
        dict(name="layer_8b", kind="layer", tokens=16384, adapters=4, rank=16, hidden=4096, kv=1024, mlp=14336, p=0.1, base="bf16"),
        # a 70B-class decoder layer with NF4 base weights
        dict(name="layer_70b_nf4", kind="layer", tokens=8192, adapters=6, rank=64, hidden=8192, kv=1024, mlp=28672, p=0.1, base="nf4"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A multiple of 128, over the logarithm: powers of two and odd multiples alike."""
    return 128 * _log_int(rng, lo // 128, hi // 128)


def draw(rng: random.Random):
    kind = rng.choice(["evaluate", "evaluate", "train", "train", "train", "packed", "packed", "nf4", "dequant", "norm_act", "layer"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    p = rng.choice([0.0, 0.05, 0.1])
    if kind == "evaluate":
        return dict(kind=kind, tokens=_log_int(rng, 1, 4096), k=_width(rng, 1024, 14336), n=_width(rng, 1024, 14336),
                    rank=rng.choice([8, 16, 32, 64, 128]), dtype=dtype, bias=rng.random() < 0.5)
    if kind == "train":
        return dict(kind=kind, tokens=_log_int(rng, 100, 8192), k=_width(rng, 1024, 8192), n=_width(rng, 1024, 14336),
                    rank=rng.choice([8, 16, 32, 64, 128]), p=p, dtype=dtype, bias=rng.random() < 0.3,
                    mask=rng.choice(["drawn", "drawn", "given"]))
    if kind == "packed":
        return dict(kind=kind, tokens=_log_int(rng, 500, 16384), adapters=rng.randint(2, 8), ranks=rng.choice(["16", "32", "64", "mixed"]),
                    k=_width(rng, 1024, 8192), n=_width(rng, 1024, 14336), p=p, dtype=dtype)
    if kind == "nf4":
        return dict(kind=kind, tokens=_log_int(rng, 128, 8192), k=_width(rng, 2048, 8192), n=_width(rng, 2048, 14336),
                    rank=rng.choice([8, 16, 32, 64]), p=p, dtype=dtype)
    if kind == "dequant":
        return dict(kind=kind, k=_width(rng, 1024, 8192), n=_width(rng, 1024, 28672), blocksize=rng.choice([64, 64, 128, 256]),
                    nested=rng.random() < 0.75, dtype=dtype)
    if kind == "norm_act":
        return dict(kind=kind, tokens=_log_int(rng, 100, 16384), hidden=_width(rng, 1024, 8192), mlp=_width(rng, 2048, 14336),
                    train_norm=rng.random() < 0.5, dtype=dtype)
    return dict(kind=kind, tokens=_log_int(rng, 1024, 12288), adapters=rng.randint(1, 6), rank=rng.choice([8, 16, 32, 64]),
                hidden=_width(rng, 2048, 5120), kv=rng.choice([512, 1024]), mlp=_width(rng, 4096, 14336), p=p,
                base=rng.choice(["bf16", "nf4"]))


# ---------------------------------------------------------------------------------------------------- inputs


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _adapter(g, k, n, r, dtype):
    """A and B as they are in the middle of a run: A ~ kaiming-uniform(a = sqrt 5), B small."""
    a = ((torch.rand(r, k, generator=g, device=DEV) * 2 - 1) / k ** 0.5).to(dtype)
    return a.requires_grad_(), _randn(g, n, r, std=0.01, dtype=dtype).requires_grad_()


def _segments(tokens, adapters):
    """Tokens of each adapter in a packed batch: sample lengths of a log-normal distribution, dealt to the adapters in
    turn.  Every adapter gets some.  (A function of the case: the padded batch of a case has one shape.)"""
    rng = random.Random(1000 * tokens + adapters)
    median = tokens / (4 * adapters)
    per, left, i = [0] * adapters, tokens, 0
    while left > 0:
        n = max(1, min(int(median * rng.lognormvariate(0.0, 0.8)), left))
        if i < adapters:
            n = min(n, max(1, left // (adapters - i)))   # (the adapters behind this one get tokens too)
        per[i % adapters] += n
        left -= n
        i += 1
    return per


def _rank_list(ranks, adapters):
    return ([8, 16, 32, 64] * adapters)[:adapters] if ranks == "mixed" else [int(ranks)] * adapters


def _drops(p, adapters):
    """Dropout rates around the case's: one adapter without, the others with p or half of it."""
    return ([0.0, p / 2, p, p] * adapters)[:adapters] if adapters > 1 else [p]


def _scales(adapters):
    return ([1.0, 2.0, 2.0, 4.0] * adapters)[:adapters]


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind = case["kind"]
    s = {"case": dict(case), "seed": seed}
    dtype = DTYPES[case.get("dtype", "bf16")]
    if kind in ("evaluate", "train", "packed", "nf4"):
        k, n = case["k"], case["n"]
        w = _randn(g, n, k, std=0.02, dtype=dtype)
    if kind in ("evaluate", "train", "nf4"):
        m = case["tokens"]
        s["x"] = _randn(g, m, k, dtype=dtype)
        s["a"], s["b"] = _adapter(g, k, n, case["rank"], dtype)
        s["alpha"] = 2.0
    if kind in ("evaluate", "train"):
        s["w"] = w
        s["bias"] = _randn(g, n, std=0.1, dtype=dtype) if case["bias"] else None
    if kind in ("train", "nf4"):
        s["x"].requires_grad_()
        s["dy"] = _randn(g, m, n, dtype=dtype)
        s["mask"] = (torch.rand(m, k, generator=g, device=DEV) >= case["p"]) if case.get("mask") == "given" and case["p"] > 0 else None
    if kind == "nf4":
        s["packed"], s["quant"] = quantize_nf4(w)
    if kind == "packed":
        seq, ranks = _segments(case["tokens"], case["adapters"]), _rank_list(case["ranks"], case["adapters"])
        s["info"] = info = prepare_multi_lora_batch_info(seq, list(range(len(seq))), ranks, _drops(case["p"], len(seq)), _scales(len(seq)), BLOCK)
        rows = sum(info.padded_seq_len_list)
        s["w"] = w
        s["x"] = _randn(g, 1, rows, k, dtype=dtype).requires_grad_()
        s["dy"] = _randn(g, 1, rows, n, dtype=dtype)
        ab = [_adapter(g, k, n, r, dtype) for r in ranks]
        s["a"], s["b"] = [a for a, _ in ab], [b for _, b in ab]
    if kind == "dequant":
        s["packed"], s["quant"] = quantize_nf4(_randn(g, case["n"], case["k"], std=0.02, dtype=dtype), blocksize=case["blocksize"],
                                               compress_statistics=case["nested"])
    if kind == "norm_act":
        m, h, i = case["tokens"], case["hidden"], case["mlp"]
        s["x"] = _randn(g, m, h, dtype=dtype).requires_grad_()
        s["w"] = (1 + 0.1 * torch.randn(h, generator=g, device=DEV)).to(dtype).requires_grad_(case["train_norm"])
        s["dy"] = _randn(g, m, h, dtype=dtype)
        s["gate_up"] = _randn(g, m, 2 * i, dtype=dtype).requires_grad_()
        s["dc"] = _randn(g, m, i, dtype=dtype)
    if kind == "layer":
        _prepare_layer(s, g, case, seed)
    return s


def _prepare_layer(s, g, case, seed):
    h, kv, mlp, n_ad, r = case["hidden"], case["kv"], case["mlp"], case["adapters"], case["rank"]
    drops, scales = _drops(case["p"], n_ad), _scales(n_ad)
    layer = DecoderLayerLoRAProjections.from_shapes(
        h, kv, mlp, {f"lora_{i}": (r, scales[i] * r, drops[i]) for i in range(n_ad)}, device=DEV, seed=seed)
    for lin in layer.linears().values():
        for name in lin.lora_A:
            with torch.no_grad():
                lin.lora_A[name].weight.copy_((torch.rand(r, lin.in_features, generator=g, device=DEV) * 2 - 1) / lin.in_features ** 0.5)
                lin.lora_B[name].weight.copy_(torch.randn(lin.out_features, r, generator=g, device=DEV) * 0.01)
        if case["base"] == "nf4":
            packed, state = quantize_nf4(lin.base_layer.weight.detach())
            packed = torch.nn.Parameter(packed, requires_grad=False)
            packed.quant_state = state
            lin.base_layer.weight = packed
    layer.train()
    seq = _segments(case["tokens"], n_ad)
    info = prepare_multi_lora_batch_info(seq, list(range(n_ad)), [r] * n_ad, drops, scales, BLOCK, allow_empty_micro_batch_info=True)
    rows = sum(info.padded_seq_len_list)
    s.update(layer=layer, info=info)
    # the residual stream before each norm, attention's output, and the gradients that come back from attention, the
    # output projection's consumer and the layer's end (attention and the residual additions are the caller's)
    s["hidden"], s["ctx"], s["mid"] = (_randn(g, 1, rows, h).requires_grad_() for _ in range(3))
    s["norm1"], s["norm2"] = ((1 + 0.1 * torch.randn(h, generator=g, device=DEV)).bfloat16() for _ in range(2))
    s["dqkv"], s["do"], s["dout"] = _randn(g, 1, rows, h + 2 * kv), _randn(g, 1, rows, h), _randn(g, 1, rows, h)
    s["leaves"] = [s["hidden"], s["ctx"], s["mid"]] + [m[name].weight for lin in layer.linears().values()
                                                       for m in (lin.lora_A, lin.lora_B) for name in m]


# ---------------------------------------------------------------------------------------------------- one pass


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "evaluate":
        with torch.no_grad():
            return fused_linear_lora(s["x"], s["w"], s["a"], s["b"], s["alpha"], linear_bias=s["bias"])
    if kind == "train":
        y = fused_linear_lora(s["x"], s["w"], s["a"], s["b"], s["alpha"], seed=s["seed"], dropout_p=case["p"], linear_bias=s["bias"],
                              dropout_mask=s["mask"])
        return (y.detach(), *torch.autograd.grad(y, (s["x"], s["a"], s["b"]), s["dy"]))
    if kind == "nf4":
        y = fused_linear_lora_nf4(s["x"], s["packed"], s["quant"], s["a"], s["b"], s["alpha"], seed=s["seed"], dropout_p=case["p"])
        return (y.detach(), *torch.autograd.grad(y, (s["x"], s["a"], s["b"]), s["dy"]))
    if kind == "packed":
        i = s["info"]
        y = fused_linear_multi_lora(
            s["x"], s["w"], lora_a_list=s["a"], lora_b_list=s["b"], seq_len_list=i.seq_len_list, padded_seq_len_list=i.padded_seq_len_list,
            block_to_lookup_table=i.block_to_lookup_table, block_to_dropout_p=i.block_to_dropout_p, block_to_alpha=i.block_to_alpha,
            enable_dropout=i.enable_dropout, same_dropout_p_value=i.same_dropout_p_value, max_r=i.max_r, seed=s["seed"],
            routing=i.routing(enable_dropout=i.enable_dropout))
        return (y.detach(), *torch.autograd.grad(y, (s["x"], *s["a"], *s["b"]), s["dy"]))
    if kind == "dequant":
        return dequantize_nf4_triton(s["packed"], s["quant"])
    if kind == "norm_act":
        y, c = rms_norm(s["x"], s["w"], 1e-5), silu_mul_merged(s["gate_up"])
        wrt = (s["x"], s["gate_up"]) + ((s["w"],) if s["w"].requires_grad else ())
        return (y.detach(), c.detach(), *torch.autograd.grad((y, c), wrt, (s["dy"], s["dc"])))
    return _run_layer(s)


def _run_layer(s):
    manager = multi_lora.get_multi_lora_manager()
    if manager is None:
        manager = multi_lora.init_multi_lora_manager([None] * 32, 1, None, [1] * 32)
    manager.clear_batch_info()
    manager.add_batch_info(s["info"])
    random.seed(s["seed"])   # the layer draws its dropout seeds from Python's generator: seeded, the pass is reproducible
    lin = s["layer"].linears()
    qkv = lora_forward(lin["qkv"], rms_norm(s["hidden"], s["norm1"], 1e-5))
    o = lora_forward(lin["o"], s["ctx"])
    gate_up = lora_forward(lin["gate_up"], rms_norm(s["mid"], s["norm2"], 1e-5))
    out = swiglu_lora_forward(lin["down"], gate_up)
    return (qkv.detach(), o.detach(), out.detach(), *torch.autograd.grad((qkv, o, out), s["leaves"], (s["dqkv"], s["do"], s["dout"])))


# ------------------------------------------------------------------------------------------- what a pass must do


def _linear_work(m, k, n, r, w_bytes, train):
    """Real tokens m; r: the rank each token is multiplied with, summed adapters' r for the adapter tensors."""
    flops, bytes_ = 2.0 * m * k * n + 2.0 * m * r * (k + n), 2.0 * m * (k + n) + w_bytes
    if train:   # dX = dY W + dS A, dS = dY B, dA = dS^T X, dB = dY^T S; X and dY read, dX written
        flops += 2.0 * m * k * n + 4.0 * m * r * (k + n)
        bytes_ += 2.0 * m * (k + n)
    return flops, bytes_


def _nf4_bytes(elems, blocksize=64, nested=True):
    return elems / 2 + (elems / blocksize + 4.0 * elems / (blocksize * 256) if nested else 4.0 * elems / blocksize)


def work(case):
    kind = case["kind"]
    if kind in ("evaluate", "train", "nf4"):
        k, n, r, m, train = case["k"], case["n"], case["rank"], case["tokens"], kind != "evaluate"
        flops, bytes_ = _linear_work(m, k, n, r, _nf4_bytes(k * n) if kind == "nf4" else 2.0 * k * n, train)
        bytes_ += 2.0 * r * (k + n) * (2 if train else 1) + (m * k if case.get("mask") == "given" and case.get("p") else 0)
        return {"bytes": bytes_, "flops": flops}
    if kind == "packed":
        k, n, ranks = case["k"], case["n"], _rank_list(case["ranks"], case["adapters"])
        flops, bytes_ = _linear_work(case["tokens"], k, n, sum(ranks) / len(ranks), 2.0 * k * n, True)
        return {"bytes": bytes_ + 4.0 * sum(ranks) * (k + n), "flops": flops}
    if kind == "dequant":
        elems = case["k"] * case["n"]
        return {"bytes": 2.0 * elems + _nf4_bytes(elems, case["blocksize"], case["nested"]), "flops": 1.0 * elems}
    if kind == "norm_act":
        m, h, i = case["tokens"], case["hidden"], case["mlp"]
        return {"bytes": 2.0 * m * (5 * h + 8 * i), "flops": 20.0 * m * (h + i)}
    h, kv, mlp, r, m = case["hidden"], case["kv"], case["mlp"], case["rank"], case["tokens"]
    flops = bytes_ = 0.0
    for k, n in ((h, h + 2 * kv), (h, h), (h, 2 * mlp), (mlp, h)):
        f, b = _linear_work(m, k, n, r, _nf4_bytes(k * n) if case["base"] == "nf4" else 2.0 * k * n, True)
        flops += f
        bytes_ += b + 4.0 * case["adapters"] * r * (k + n)
    return {"bytes": bytes_ + 2.0 * m * 10 * h, "flops": flops}


def tolerance(case):
    # Dequantisation is bit-exact.  Everything else rounds 16-bit results of fp32 sums.  Measured against fp64: outputs
    # and dX 1.7e-3 (bf16) / 2.1e-4 (fp16) of their norm, gradients through the stored 16-bit rank-r intermediates 2.4e-3 /
    # 3.0e-4; a layer's outputs with its sums in another order differ by 1.0e-3 of each other.  About four times that.
    if case["kind"] == "dequant":
        return "exact"
    return {"rel": 0.0012 if case.get("dtype") == "fp16" else 0.01}
