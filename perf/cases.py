"""The work that programs on this framework have it do, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" names the entry point:

  linear   llama.qlinear.QuantLinear.forward, the layer loaded as a loader does (repacked where the library recommends it)
  vecquant quant_cuda.vecquant{3,4}matmul_cherryq over the checkpoint buffers: the drop-in operator, fp16 or fp32 tensors
  steps    CherryLlamaDecoder.step_logits: one captured token step per token (decoding, per-token perplexity)
  prompt   CherryLlamaDecoder.prefill: the whole prompt in one pass
  qat      one forward and backward of the training-side llama.cherry_linear.QuantLinear
  convert  a trained weight packed, repacked into the weight stream, and unpacked to the dense weight
"""
import math
import os
import sys

import torch

_PKG = os.path.abspath("mixed-precision-cuda-kernel_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import cherryq_decoder  # noqa: E402
import quant_cuda  # noqa: E402
from llama.cherry_linear import QuantLinear as TrainLinear  # noqa: E402
from llama.qlinear import QuantLinear  # noqa: E402
from llama.quantizer import FullSymQuantizer  # noqa: E402

FRACTION = 1 / 256  # share of the input channels kept in high precision
_DTYPES = {"float16": torch.float16, "float32": torch.float32, "bfloat16": torch.bfloat16}
_LLAMA_7B = dict(bits=4, group=128, hidden=4096, inter=11008, layers=32, heads=32, kv_heads=32, vocab=32000, max_pos=256)


def listed():
    return [
        # one decoded token through one attention projection of a 7B model: the smallest call there is
        dict(name="linear_row1_w4_4096x4096", kind="linear", bits=4, group=128, k=4096, n=4096, rows=1),
        # the drop-in operator as a program written for it calls it, one token, 7B gate / up and down
        dict(name="vecquant_row1_w4_4096x11008", kind="vecquant", bits=4, group=128, k=4096, n=11008, rows=1, dtype="float16"),
        dict(name="vecquant_row1_w3_11008x4096", kind="vecquant", bits=3, group=128, k=11008, n=4096, rows=1, dtype="float16"),
        # the operator's own micro-benchmark: 16 rows of fp32 tensors over a 3-bit 13B-wide layer
        dict(name="vecquant_rows16_f32_w3_4096x13824", kind="vecquant", bits=3, group=128, k=4096, n=13824, rows=16, dtype="float32"),
        # a few sequences decoded together: 13B gate / up in 3 bits, 70B gate / up in 4
        dict(name="linear_rows8_w3_5120x13824", kind="linear", bits=3, group=128, k=5120, n=13824, rows=8),
        dict(name="linear_rows16_w4_8192x28672", kind="linear", bits=4, group=128, k=8192, n=28672, rows=16),
        # a short prompt of odd length, and a prompt of the evaluation's full length
        dict(name="linear_rows99_w4_4096x11008", kind="linear", bits=4, group=128, k=4096, n=11008, rows=99),
        dict(name="linear_rows2048_w4_4096x11008", kind="linear", bits=4, group=128, k=4096, n=11008, rows=2048),
        # a whole 7B model: decoding token by token, and its 128-token prompt
        dict(name="steps32_7b_w4", kind="steps", tokens=32, **_LLAMA_7B),
        dict(name="prompt128_7b_w4", kind="prompt", tokens=128, **_LLAMA_7B),
        # quantisation-aware training of one 7B layer on a 2048-token document
        dict(name="qat_bf16_rows2048_w4_4096x11008", kind="qat", bits=4, group=128, k=4096, n=11008, rows=2048, dtype="bfloat16"),
        # a checkpoint made and loaded, layer by layer
        dict(name="convert_w3_5120x13824", kind="convert", bits=3, group=128, k=5120, n=13824),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "vecquant", "vecquant", "steps", "prompt", "qat", "convert"])
    bits = rng.choice([3, 4])
    if kind in ("steps", "prompt"):
        heads = rng.randint(8, 64)
        # the reference models' proportions: MLP about 2.7 times the width, full or grouped key / value heads
        kv = rng.choice([heads, heads, next(d for d in (8, 4, 2, 1) if heads % d == 0)])
        tokens = _log(rng, 8, 32) if kind == "steps" else _log(rng, 8, 600)
        c = dict(kind=kind, tokens=tokens, bits=bits, group=128, hidden=128 * heads, inter=_log(rng, 256 * heads, 448 * heads, 8),
                 layers=rng.randint(1, 4), heads=heads, kv_heads=kv, vocab=32000, max_pos=max(tokens, rng.choice([256, 1024, 2048])))
        return c
    c = dict(kind=kind, bits=bits, group=128, k=_log(rng, 1024, 28672, 8), n=_log(rng, 512, 28672, 8))
    if kind == "linear":
        c["rows"] = _log(rng, 1, 2048)
        while c["k"] * c["n"] > 8192 * 28672:
            c["n"] = _log(rng, 512, 28672, 8)
    elif kind == "vecquant":
        c["dtype"] = rng.choice(["float16", "float16", "float32"]) if bits == 3 else "float16"
        c["rows"] = _log(rng, 1, 32)
        if bits == 3 and rng.random() < 0.25:
            c["group"] = 64
    elif kind == "qat":
        c["k"], c["n"] = _log(rng, 1024, 11008, 8), _log(rng, 512, 11008, 8)
        c["rows"], c["dtype"] = _log(rng, 128, 2048), rng.choice(["float16", "bfloat16", "float32"])
    else:
        c["k"], c["n"] = _log(rng, 1024, 16000, 8), _log(rng, 512, 16000, 8)
    return c


def _cherries(k):
    return math.ceil(k * FRACTION) // 8 * 8


def _weight(case, gen, dtype=torch.float16):
    """A weight as trained: N(0, 0.02), the channels that matter ten times as large, and those channels."""
    k, n = case["k"], case["n"]
    w = torch.randn((n, k), device="cuda", generator=gen, dtype=torch.float32) * 0.02
    idx = torch.randperm(k, device="cuda", generator=gen)[:_cherries(k)].sort().values
    w[:, idx] *= 10
    return w.to(dtype), idx


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, bits, group = case["kind"], case["bits"], case["group"]
    state = dict(case)
    if kind in ("steps", "prompt"):
        cfg = cherryq_decoder.DecoderConfig(
            hidden_size=case["hidden"], intermediate_size=case["inter"], num_hidden_layers=case["layers"],
            num_attention_heads=case["heads"], num_key_value_heads=case["kv_heads"], vocab_size=case["vocab"],
            max_position_embeddings=case["max_pos"], w_bits=bits, group_size=group, cherry_fraction=FRACTION)
        model = cherryq_decoder.CherryLlamaDecoder(cfg, seed=seed)
        model.prepack()
        if kind == "steps":
            model.capture()
        state.update(model=model, ids=torch.randint(0, case["vocab"], (case["tokens"],), device="cuda", generator=gen))
        return state
    k, n = case["k"], case["n"]
    if kind == "qat":
        dtype = _DTYPES[case["dtype"]]
        w, idx = _weight(case, gen, dtype)
        with torch.device("cuda"):
            lin = TrainLinear(k, n, bias=False, w_bits=bits, group_size=group, cherryq=True, cherry_fraction=FRACTION).to(dtype)
        lin.weight.data.copy_(w)
        lin.register_cherry_indices(idx)
        lin.train()
        x = torch.randn((case["rows"], k), device="cuda", generator=gen).to(dtype).requires_grad_()
        # the loss's gradient, averaged over the tokens and scaled as half-precision training scales it
        gy = (torch.randn((case["rows"], n), device="cuda", generator=gen) * 0.01).to(dtype)
        state.update(lin=lin, x=x, gy=gy)
        return state
    w, idx = _weight(case, gen)
    if kind == "convert":
        state.update(weight=w, idx=idx)
        return state
    cherry_indices, cherry_weight, qweight, scales = quant_cuda.pack_cherryq(bits, w, idx, group)
    del w
    x = torch.randn((case["rows"], k), device="cuda", generator=gen)
    if kind == "linear":
        with torch.device("cuda"):
            q = QuantLinear(bits, group, FullSymQuantizer, FRACTION, k, n, bias=False)
        q.cherry_indices, q.cherry_weight, q.qweight, q.scales = cherry_indices, cherry_weight, qweight, scales
        if quant_cuda.prepack_recommended(bits, k, n, q.num_cherries, group):
            q.prepack()
        state.update(lin=q, x=x.half())
        return state
    dtype = _DTYPES[case["dtype"]]
    f32 = dtype == torch.float32
    state.update(x=x.to(dtype), qweight=qweight, cherry_weight=cherry_weight.to(dtype), scales=scales.to(dtype),
                 cherry_indices=cherry_indices.to(torch.int32 if f32 else torch.int16))
    return state


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return s["lin"](s["x"])
    if kind == "vecquant":
        mul = torch.zeros((s["rows"], s["n"]), dtype=s["x"].dtype, device="cuda")
        args = (s["x"], s["qweight"], s["cherry_weight"], s["cherry_indices"], s["scales"], mul, s["group"])
        if s["bits"] == 4:
            quant_cuda.vecquant4matmul_cherryq(*args)
        else:
            quant_cuda.vecquant3matmul_cherryq(*args, s["dtype"] == "float16")
        return mul
    if kind == "steps":
        m, t = s["model"], s["tokens"]
        return m.step_logits(s["ids"], use_graph=True), m.k_cache[:, :, :t], m.v_cache[:, :, :t]
    if kind == "prompt":
        m, t = s["model"], s["tokens"]
        return m.prefill(s["ids"]), m.k_cache[:, :, :t], m.v_cache[:, :, :t]
    if kind == "qat":
        lin, x = s["lin"], s["x"]
        x.grad = lin.weight.grad = None
        out = lin(x)
        out.backward(s["gy"])
        return out.detach(), x.grad, lin.weight.grad
    idx, cw, qw, sc = quant_cuda.pack_cherryq(s["bits"], s["weight"], s["idx"], s["group"])
    stream = quant_cuda.prepack_cherryq(s["bits"], qw, cw, idx, sc, s["k"], s["group"])
    dense = quant_cuda.unpack_cherryq(s["bits"], qw, cw, idx, sc, s["k"], s["group"])
    return idx, cw, qw, sc, stream, dense


def _packed_bytes(bits, group, k, n, io=2):
    c = _cherries(k)
    kn = k - c
    return kn // 8 * bits * n + (-(-kn // group) + c) * n * io + c * io


def work(case):
    kind, bits, group = case["kind"], case["bits"], case["group"]
    if kind in ("steps", "prompt"):
        h, i, t, v = case["hidden"], case["inter"], case["tokens"], case["vocab"]
        kv = case["kv_heads"] * (h // case["heads"])
        shapes = [(h, h), (h, kv), (h, kv), (h, h), (h, i), (h, i), (i, h)]
        weights = case["layers"] * sum(_packed_bytes(bits, group, a, b) for a, b in shapes)
        macs = case["layers"] * sum(a * b for a, b in shapes)
        pairs = t * (t + 1) // 2  # (query, key) pairs under the causal mask
        cache = case["layers"] * 2 * kv * 2  # bytes of one position's keys and values
        if kind == "steps":
            return {"bytes": t * (weights + v * h * 2 + h * 2 + v * 4) + cache * (pairs + t),
                    "flops": 2 * t * (macs + v * h) + 4 * case["layers"] * h * pairs}
        return {"bytes": weights + t * h * 2 + v * h * 2 + v * 4 + cache * t,
                "flops": 2 * (t * macs + v * h) + 4 * case["layers"] * h * pairs}
    k, n = case["k"], case["n"]
    if kind == "convert":
        return {"bytes": 2 * n * k + 2 * _packed_bytes(bits, group, k, n) + 2 * n * k, "flops": 4 * n * k}
    rows = case["rows"]
    if kind == "qat":
        size = 4 if case["dtype"] == "float32" else 2
        # weight, input and output's gradient in; output, input's and weight's gradients out
        return {"bytes": size * (2 * n * k + 2 * rows * k + 2 * rows * n), "flops": 3 * 2 * rows * k * n}
    size = 4 if case.get("dtype") == "float32" else 2
    return {"bytes": _packed_bytes(bits, group, k, n, size) + size * rows * (k + n), "flops": 2 * rows * k * n}


def tolerance(case):
    kind = case["kind"]
    if kind == "convert":
        return "exact"
    if kind in ("steps", "prompt"):
        return {"rel": 2e-2}  # fp16 activations through a chain of layers: what the same model in dense fp16 differs by
    if case.get("dtype") == "float32":
        return {"rel": 1e-5}
    if case.get("dtype") == "bfloat16":
        return {"rel": 1e-2}
    return {"rel": 1e-3}  # fp16 results, and weights rounded to fp16 or not before the product
