"""The performance cases of hot_amd: the work that a training program has the framework do, through
its public entry points, from a handful of tokens to the largest layers.

Kinds of case (field "kind"):

  backward   ops.linear_backward, the fused HOT backward of one linear layer: g_x and g_W from g_y, W and the
             saved activation buffer (what bench.py measures)
  buffer     ops.abc_forward, the INT8 activation buffer that the forward pass saves
  rowwise    ops.hq_rowwise, the block-Hadamard quantiser alone (the kernel-level sweep of bench.py)
  op         HLQ_backward.backward, the drop-in op, at the sizes of its latency harness
  step       a training step (forward and backward through autograd) of one HQ_Linear, or of two with a GELU
             between them (the MLP of a transformer block), on 2-D or 3-D activations

Fields: L tokens (B samples of T tokens in 3-D steps), O outputs, I inputs of the layer; dtype of g_y, W, x and
the results; rule: how the low-rank projection along the tokens is chosen ("python": from the token count, blocks of
up to 8192 tokens; "paper": blocks of 16, the 8 lowest sequencies); bits of the g_x operands; rounding and scale
(one quantiser step per tensor or per token).
"""
import math

import torch
import torch.nn as nn

from hot_amd import HLQ_backward, args, ops
from hot_amd.hadamard_matmul import hla_rows, paper_rows, run_major
from hot_amd.quant_matmul import HQ_Linear

_DT = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_SIZE = {"fp32": 4, "bf16": 2, "fp16": 2}


def listed():
    return [
        # the reference's latency harness (measure.py) on the drop-in op: 49 tokens, fp32, a step per token
        dict(name="op_49_tokens", kind="op", L=49, O=3072, I=768, dtype="fp32", scale="row"),
        # a classification head: one token per image of a batch of 128, 100 classes (widths of the SAWB recipe are
        # multiples of 8), stochastic per-tensor quantisers
        dict(name="head_step", kind="step", B=0, T=128, I=768, H=0, O=100, dtype="bf16", recipe="stoch", bias=True),
        # odd sizes: a token count that no power of two divides, widths that fill no tile, fp16
        dict(name="ragged_backward", kind="backward", L=3003, O=1000, I=520, dtype="fp16", rule="python", bits=4,
             rounding="nearest", scale="tensor"),
        # ViT-B layers at 64 x 197 tokens: fc1 (the headline benchmark), qkv in full precision inputs, fc2 with the
        # stochastic per-token INT8 quantisers
        dict(name="vit_fc1_backward", kind="backward", L=12608, O=3072, I=768, dtype="bf16", rule="python", bits=4,
             rounding="nearest", scale="tensor"),
        dict(name="vit_qkv_backward_fp32", kind="backward", L=12608, O=2304, I=768, dtype="fp32", rule="python", bits=4,
             rounding="nearest", scale="tensor"),
        dict(name="vit_fc2_backward_int8", kind="backward", L=12608, O=768, I=3072, dtype="bf16", rule="python", bits=8,
             rounding="stoch", scale="row"),
        # the activation buffer of fc2 (its input is the widest of the block), saved in forward
        dict(name="vit_fc2_buffer", kind="buffer", L=12608, O=768, I=3072, dtype="bf16", rule="python", scale="tensor"),
        # the quantiser alone: 16384 rows of 4096, blocks of 32, packed INT4, a step per row
        dict(name="rowwise_16384", kind="rowwise", L=16384, O=4096, dtype="bf16", block=32, bits=4, rounding="nearest",
             scale="row"),
        # attention projection with the reference's treatment of 3-D activations: every image of 197 tokens has its
        # own quantiser steps
        dict(name="proj_step_per_sample", kind="step", B=64, T=197, I=768, H=0, O=768, dtype="bf16", recipe="stoch",
             bias=True),
        # the MLP of a ViT-B block at batch 128, tokens flattened, the training recipe (per-token stochastic g_y, SAWB)
        dict(name="mlp_step", kind="step", B=0, T=25216, I=768, H=3072, O=768, dtype="bf16", recipe="canonical", bias=True),
        # Llama-7B layers at 8192 tokens: gate/up with blocks of 16 tokens, down with one block of 8192
        dict(name="llama_gate_up_backward", kind="backward", L=8192, O=11008, I=4096, dtype="bf16", rule="paper", bits=4,
             rounding="nearest", scale="tensor"),
        dict(name="llama_down_backward_8192", kind="backward", L=8192, O=4096, I=11008, dtype="bf16", rule="python", bits=4,
             rounding="nearest", scale="tensor"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, of):
    return max(of, _log_int(rng, lo, hi) // of * of)


def _tokens(rng, lo, hi):
    # token counts as they occur: anything, images of 197 tokens, and sequences whose length holds a power of two
    how = rng.randrange(4)
    if how == 0:
        return max(lo, _log_int(rng, lo, hi) | 1)
    if how == 1:
        return 197 * max(1, _log_int(rng, lo, hi) // 197)
    return _multiple(rng, max(lo, 64), hi, rng.choice((8, 16, 64, 128, 256, 1024)))


def draw(rng):
    kind = rng.choice(("backward",) * 5 + ("step",) * 3 + ("buffer", "rowwise", "rowwise", "op"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp32", "fp16"))
    rounding, scale = rng.choice(("nearest", "nearest", "stoch")), rng.choice(("tensor", "row"))
    if kind == "backward":
        while True:
            L = _tokens(rng, 64, 16384)
            O, I = _multiple(rng, 64, 11008, rng.choice((8, 16, 128))), _multiple(rng, 64, 11008, rng.choice((8, 16, 128)))
            # no larger than the largest listed case, and within what one call takes
            if L * O * I <= 8192 * 11008 * 4096 and L * (O + I) <= 8192 * 15104:
                break
        rule = rng.choice(("python", "python", "paper"))
        return dict(kind=kind, L=L, O=O, I=I, dtype=dtype, rule=rule, bits=rng.choice((4, 4, 8)), rounding=rounding, scale=scale)
    if kind == "step":
        recipe, dtype = rng.choice(("canonical", "stoch", "nearest")), rng.choice(("bf16", "bf16", "fp32"))
        three_d, mlp = rng.random() < 0.4, rng.random() < 0.35
        B = rng.randrange(4, 129) if three_d else 0
        while True:
            T = rng.choice((49, 64, 196, 197, 208)) if three_d else _tokens(rng, 64, 25216)
            I, O = _multiple(rng, 192, 1024, 8), _multiple(rng, 96, 3072, 8 if recipe == "canonical" else 4)
            macs = (B or 1) * T * I * (8 * I if mlp else O)
            if macs <= 25216 * 768 * 6144 / (8 if dtype == "fp32" else 1):      # the plain forward product in fp32 is slow
                break
        return dict(kind=kind, B=B, T=T, I=I, H=4 * I if mlp else 0, O=I if mlp else O, dtype=dtype, recipe=recipe,
                    bias=rng.random() < 0.75)
    if kind == "buffer":
        return dict(kind=kind, L=_tokens(rng, 256, 25216), O=0, I=_multiple(rng, 256, 4096, 8), dtype=dtype,
                    rule=rng.choice(("python", "python", "paper")), scale=rng.choice(("tensor", "tensor", "sawb")))
    if kind == "rowwise":
        while True:
            L, O = _log_int(rng, 1000, 65536), _multiple(rng, 256, 11008, 64)
            if L * O * _SIZE[dtype] <= 65536 * 4096 * 4:
                break
        return dict(kind=kind, L=L, O=O, dtype=dtype, block=rng.choice((16, 32, 64)), bits=rng.choice((4, 8)), rounding=rounding,
                    scale=rng.choice(("row", "row", "tensor")))
    return dict(kind="op", L=_log_int(rng, 16, 512), O=_multiple(rng, 256, 4096, 16), I=_multiple(rng, 256, 4096, 8),
                dtype=rng.choice(("fp32", "bf16")), scale=scale)


# ---- inputs ---------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _activations(g, shape, dtype):
    # what leaves a layer norm
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _gradient(g, shape, dtype):
    # output gradients: N(0, 1e-3), one entry in a hundred fifty times larger
    v = torch.randn(shape, generator=g, device="cuda") * 1e-3
    return torch.where(torch.rand(shape, generator=g, device="cuda") < 0.01, v * 50, v).to(dtype)


def _weight(g, O, I, dtype):
    return ((torch.rand(O, I, generator=g, device="cuda") * 2 - 1) / I ** 0.5).to(dtype)


def _rule(case):
    L = case["L"]
    if case["rule"] == "paper":
        return (1, [0]) if L % 16 else paper_rows(16, 8)
    n, rows = hla_rows(L)
    if n > 8192:
        n, rows = hla_rows(8192)
    return (n, run_major(rows)) if n > 128 else (n, rows)


def _options(case, seed):
    n, rows = _rule(case)
    bits, rounding, scale = case.get("bits", 4), case.get("rounding", "nearest"), case["scale"]
    act = "sawb" if case["kind"] == "buffer" and scale == "sawb" else "tensor"
    step = "row" if scale == "row" else "tensor"
    n_o = min(16, case["O"] & -case["O"]) if case["O"] else 16
    return ops.HotOptions(n_o=n_o, hla_n=int(n), hla_rows=tuple(int(v) for v in rows), gx_bits=bits, w_bits=bits,
                          gx_round=rounding, gw_round=rounding, gx_scale=step, gw_scale=step, act_scale=act, seed=int(seed) % 100003)


def _recipe(name):
    if name == "canonical":
        args.canonical_recipe()
    elif name == "stoch":
        args.hot_recipe(gx="stoch", gw="stoch")
    else:
        args.hot_recipe()
    args.layer_quant_dict.clear()


def prepare(case, seed):
    g, kind, dt = _generator(seed), case["kind"], _DT[case["dtype"]]
    if kind == "backward":
        opt = _options(case, seed)
        x = _activations(g, (case["L"], case["I"]), dt)
        xq, sx = ops.abc_forward(x, opt)
        return dict(kind=kind, gy=_gradient(g, (case["L"], case["O"]), dt), w=_weight(g, case["O"], case["I"], dt), xq=xq, sx=sx, opt=opt)
    if kind == "buffer":
        return dict(kind=kind, x=_activations(g, (case["L"], case["I"]), dt), opt=_options(case, seed))
    if kind == "rowwise":
        scale = 10.0 ** (torch.rand(case["O"], generator=g, device="cuda") * 2 - 1)
        x = (torch.randn(case["L"], case["O"], generator=g, device="cuda") * scale).to(dt)
        return dict(kind=kind, x=x, n=case["block"], bits=case["bits"], rounding=case["rounding"], scale=case["scale"], seed=int(seed) % 100003)
    if kind == "op":
        def lognormal(r, c):
            return torch.exp(1.0 + 0.1 * torch.randn(r, c, generator=g, device="cuda")).to(dt)
        return dict(kind=kind, gy=lognormal(case["L"], case["O"]), w=lognormal(case["O"], case["I"]),
                    x=lognormal(case["L"], case["I"]), per_token=case["scale"] == "row")
    _recipe(case["recipe"])
    dims = (case["I"], case["H"], case["O"]) if case["H"] else (case["I"], case["O"])
    layers = []
    for a, b in zip(dims, dims[1:]):
        lin = HQ_Linear(a, b, bias=case["bias"]).to("cuda").to(dt)
        with torch.no_grad():
            lin.weight.copy_(_weight(g, b, a, dt))
            if case["bias"]:
                lin.bias.copy_((torch.rand(b, generator=g, device="cuda") * 0.02 - 0.01).to(dt))
        layers += [lin] if not layers else [nn.GELU(), lin]
    shape = (case["B"], case["T"]) if case["B"] else (case["T"],)
    model = nn.Sequential(*layers)
    return dict(kind=kind, model=model, params=list(model.parameters()), recipe=case["recipe"], sr=int(seed) % 100003,
                x=_activations(g, shape + (case["I"],), dt).requires_grad_(), gy=_gradient(g, shape + (case["O"],), dt))


def run(state):
    kind = state["kind"]
    if kind == "backward":
        return ops.linear_backward(state["gy"], state["w"], state["xq"], state["sx"], state["opt"])
    if kind == "buffer":
        return ops.abc_forward(state["x"], state["opt"])
    if kind == "rowwise":
        return ops.hq_rowwise(state["x"], n=state["n"], bits=state["bits"], rounding=state["rounding"], scale=state["scale"], seed=state["seed"])
    if kind == "op":
        gx, gw, _times = HLQ_backward.backward(state["gy"], state["w"], state["x"], 0, 0, 16, state["per_token"])
        return gx, gw
    _recipe(state["recipe"])
    args.sr_step = state["sr"]          # the key of the stochastic rounding: the step number of a training run
    y = state["model"](state["x"])
    return [y] + list(torch.autograd.grad(y, [state["x"]] + state["params"], state["gy"]))


# ---- what a pass cannot do without ----------------------------------------------

def _kept(case_rule, L):
    n, rows = _rule(dict(rule=case_rule, L=L))
    return L // n * len(rows)


def work(case):
    kind, e = case["kind"], _SIZE[case["dtype"]]
    if kind in ("backward", "op"):
        L, O, I = case["L"], case["O"], case["I"]
        lp = _kept(case.get("rule", "python"), L)
        saved = lp * I if kind == "backward" else L * I * e
        return {"bytes": e * (L * O + O * I + L * I + O * I) + saved, "flops": 2.0 * O * I * (L + lp)}
    if kind == "buffer":
        L, I = case["L"], case["I"]
        n, rows = _rule(case)
        return {"bytes": e * L * I + L // n * len(rows) * I, "flops": float(L * I * max(1, n.bit_length() - 1))}
    if kind == "rowwise":
        L, O = case["L"], case["O"]
        return {"bytes": e * L * O + L * O * case["bits"] // 8 + 4 * L, "flops": float(L * O * (case["block"].bit_length() - 1))}
    B, T = case["B"] or 1, case["T"]
    tokens = B * T
    dims = (case["I"], case["H"], case["O"]) if case["H"] else (case["I"], case["O"])
    pairs = list(zip(dims, dims[1:]))
    kept = B * _kept("python", T)
    weights = sum(a * b + (b if case["bias"] else 0) for a, b in pairs)
    return {"bytes": e * (2.0 * tokens * (dims[0] + dims[-1]) + 2 * weights),
            "flops": sum(2.0 * a * b * (2 * tokens + kept) for a, b in pairs)}


def tolerance(case):
    kind = case["kind"]
    # Codes: a value that falls within the rounding of its fp32 transform of a boundary between two codes takes
    # either (measured: 4 in a million against the transform in another order); steps are fp32 maxima.
    if kind in ("buffer", "rowwise"):
        return {"rel": 1e-6, "differ": 5e-5}
    # Results in fp32: the same few codes by one step each (measured against 64 bits: up to 1.8e-4).  Results in 16 bits
    # are rounded once more (measured: up to 1.6e-3).
    if kind in ("backward", "op"):
        return {"rel": 7e-4 if case["dtype"] == "fp32" else 6e-3, "max": 0.5}
    # Steps: the forward product is a plain one in the layer's type, its rounding reaches the codes of the next layer.
    return {"rel": 2e-3 if case["dtype"] == "fp32" else 1e-2, "max": 0.5}
