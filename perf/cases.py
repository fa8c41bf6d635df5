"""The work a user of this package has it do, as measurable cases.

`listed()` names fixed cases, `draw(rng)` picks further ones from the same ranges, `prepare` makes what a program holds
before the call, `run` is one pass through the public entry points, `work` the bytes and operations that the pass cannot
do without, `tolerance` how far two correct implementations may be apart.

A case's `op` is one of the operators (`linear`, `simple`, `decoupled`, `varlen`, `piecewise`) or one of the blocks
(`linfusion`, `mlla`, `rala`, `focused`, `pola`); `step` says whether a pass is a forward alone (inference) or a forward
with its backward (training).
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PACKAGE = os.path.join(os.getcwd(), "flash-bidirectional-linear-attention_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from flash_bla.layers import (FocusedLinearAttention, GeneralizedLinearAttention, MambaLikeLinearAttention,  # noqa: E402
                              PolaLinearAttention, RALALinearAttention)
from flash_bla.ops.linear_attn.decoupled import decoupled_la  # noqa: E402
from flash_bla.ops.linear_attn.fused import linear_attention  # noqa: E402
from flash_bla.ops.linear_attn.varlen import varlen_linear_attention  # noqa: E402
from flash_bla.ops.piecewise_attn.kernel import piecewise_sparse_attention  # noqa: E402
from flash_bla.ops.simple_la.fused import simple_la  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}
DENSE = ("linear", "simple", "decoupled")
BLOCKS = ("linfusion", "mlla", "rala", "focused", "pola")


def listed():
    return [
        # the smallest call: one inference forward of a few heads at full precision, all latency
        dict(name="linear_fwd_fp32_T1024", op="linear", step=False, dtype="fp32", B=2, H=4, T=1024, DK=64, DV=64),
        # a training step on short sequences: six short kernels, launches count as much as bytes
        dict(name="linear_step_fp16_T1024", op="linear", step=True, dtype="fp16", B=8, H=16, T=1024, DK=64, DV=64),
        # the package's main workload: a training step on long sequences (the largest case by bytes)
        dict(name="linear_step_fp16_T16384", op="linear", step=True, dtype="fp16", B=8, H=16, T=16384, DK=64, DV=64),
        # full-precision training with wide heads
        dict(name="linear_step_fp32_D128", op="linear", step=True, dtype="fp32", B=8, H=16, T=4096, DK=128, DV=128),
        # head dims that are no multiple of 16 bytes and an odd length, as in the package's test matrix
        dict(name="linear_step_bf16_D100", op="linear", step=True, dtype="bf16", B=8, H=16, T=4093, DK=100, DV=100),
        # packed batches of ragged sequences, both head widths that such batches are trained with
        dict(name="varlen_step_bf16_D64", op="varlen", step=True, dtype="bf16", N=64, shortest=256, longest=2048, H=16,
             DK=64, DV=64),
        dict(name="varlen_step_bf16_D128", op="varlen", step=True, dtype="bf16", N=64, shortest=256, longest=2048, H=16,
             DK=128, DV=128),
        # the decoupled operator (rotary numerator, plain denominator) on long sequences
        dict(name="decoupled_step_bf16_T16384", op="decoupled", step=True, dtype="bf16", B=2, H=16, T=16384, DK=64,
             DV=64),
        # piecewise sparse attention of a video-sized sequence (the largest case by operations)
        dict(name="piecewise_fwd_bf16_T16384", op="piecewise", step=False, dtype="bf16", B=1, H=24, T=16384, DK=128,
             DV=128, density=0.25, block=64),
        # an image-generation block at inference (guidance pair, 64 x 64 latents)
        dict(name="linfusion_fwd_fp16_4096x640", op="linfusion", step=False, dtype="fp16", B=2, side=64, dim=640,
             heads=10, sr=1),
        # a training step of a vision block: first stage (many tokens, few channels) ...
        dict(name="mlla_step_bf16_56x56x64", op="mlla", step=True, dtype="bf16", B=64, side=56, dim=64, heads=2, sr=1),
        # ... and a later stage (fewer tokens, more channels)
        dict(name="pola_step_bf16_28x28x256", op="pola", step=True, dtype="bf16", B=64, side=28, dim=256, heads=8, sr=1),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(("linear", "linear", "linear", "simple", "decoupled", "varlen", "varlen", "piecewise", "linfusion",
                     "mlla", "rala", "focused", "pola"))
    if op in DENSE:
        dtype = rng.choice(("fp16", "bf16", "fp32"))
        heads = {"linear": (32, 64, 64, 128, 0), "simple": (64, 128, 0),
                 "decoupled": (32, 64) if dtype == "fp32" else (32, 64, 128)}[op]
        DK = rng.choice(heads)
        DV = DK or rng.randint(9, 128)
        DK = DK or rng.randint(9, 128)
        B, H = rng.randint(1, 8), rng.choice((2, 4, 8, 12, 16))
        most = (160 << 20) // (BYTES[dtype] * (2 if op == "decoupled" else 1) * B * H * (DK + DV))
        return dict(op=op, step=rng.random() < 0.7, dtype=dtype, B=B, H=H, T=_log(rng, 192, min(most, 16384)), DK=DK,
                    DV=DV)
    if op == "varlen":
        longest, dtype = _log(rng, 128, 8192), rng.choice(("fp16", "bf16", "bf16", "fp32"))
        DK = rng.choice((64, 64, 128, 0))
        DV = DK or rng.randint(9, 128)
        DK = DK or rng.randint(9, 128)
        N = _log(rng, 4, max(4, min(256, (160 << 10) // (BYTES[dtype] * longest))))
        return dict(op=op, step=rng.random() < 0.7, dtype=dtype, N=N, shortest=rng.randint(1, longest // 2),
                    longest=longest, H=rng.choice((4, 8, 16)), DK=DK, DV=DV)
    if op == "piecewise":
        D = rng.choice((64, 128))
        return dict(op=op, step=False, dtype=rng.choice(("fp16", "bf16")), B=1, H=rng.randint(4, 24),
                    T=_log(rng, 1024, 16384), DK=D, DV=D, density=rng.choice((0.1, 0.15, 0.25)),
                    block=rng.choice((64, 64, 128)))
    if op == "linfusion":
        side, dim = rng.choice(((64, 320), (32, 640), (16, 1280), (32, 1280), (48, 640)))
        return dict(op=op, step=rng.random() < 0.3, dtype=rng.choice(("fp16", "bf16")), B=rng.randint(1, 4), side=side,
                    dim=dim, heads=dim // 64, sr=1)
    dim_head = 32 if op in ("mlla", "rala") else rng.choice((32, 64))
    heads = rng.choice((2, 4, 8))
    side = rng.choice((8, 14, 16, 20, 28, 32, 56))
    most = max(2, min(64, (12 << 20) // (side * side * heads * dim_head)))
    return dict(op=op, step=rng.random() < 0.7, dtype=rng.choice(("fp16", "bf16", "fp32")), B=_log(rng, 2, most),
                side=side, dim=dim_head * heads, heads=heads,
                sr=rng.choice((1, 1, 2)) if op in ("focused", "pola") else 1)


def _block(case):
    op, side, dim, heads = case["op"], case["side"], case["dim"], case["heads"]
    if op == "linfusion":
        return GeneralizedLinearAttention(dim, heads=heads, dim_head=dim // heads)
    if op == "mlla":
        return MambaLikeLinearAttention(dim, (side, side), heads)
    if op == "rala":
        return RALALinearAttention(dim, (side, side), heads)
    kind = FocusedLinearAttention if op == "focused" else PolaLinearAttention
    return kind(dim, side * side, num_heads=heads, qkv_bias=True, sr_ratio=case["sr"])


def _lengths(case):
    """Sequence lengths of a packed batch: uniform between the shortest and the longest, a property of the case."""
    g = torch.Generator().manual_seed(42)
    return torch.randint(case["shortest"], case["longest"] + 1, (case["N"],), generator=g)


def prepare(case, seed):
    dev, dtype, op = "cuda", DTYPES[case["dtype"]], case["op"]
    g = torch.Generator(device=dev).manual_seed(seed)

    def values(*shape):
        return torch.randn(shape, generator=g, device=dev).to(dtype)

    def features(*shape):
        return (F.elu(torch.randn(shape, generator=g, device=dev)) + 1).to(dtype)

    state = {"case": case}
    if op in BLOCKS:
        torch.manual_seed(seed)
        block = _block(case)
        with torch.no_grad():
            for p in block.parameters():  # parameters that start at zero have moved away from it in a trained block
                if not p.any():
                    p.add_(0.02 * torch.randn(p.shape))
        block = block.to(dev, dtype)
        if hasattr(block, "rope"):
            block.rope.float()  # the rotation table stays in fp32: it is multiplied in fp32
        block.train(case["step"])
        x = values(case["B"], case["side"] ** 2, case["dim"])
        state.update(block=block, inputs=[x], grad=values(*x.shape),
                     extra=(case["side"], case["side"]) if op in ("focused", "pola") else ())
    elif op == "varlen":
        lengths = _lengths(case)
        cu = F.pad(lengths.cumsum(0), (1, 0)).to(torch.int32).to(dev)
        T, H = int(lengths.sum()), case["H"]
        state.update(inputs=[features(T, H, case["DK"]), features(T, H, case["DK"]), values(T, H, case["DV"])],
                     grad=values(T, H, case["DV"]), cu=cu, longest=case["longest"])
    else:
        lead = (case["B"], case["H"], case["T"])
        make = values if op == "piecewise" else features
        count = 4 if op == "decoupled" else 2
        state.update(inputs=[make(*lead, case["DK"]) for _ in range(count)] + [values(*lead, case["DV"])],
                     grad=values(*lead, case["DV"]))
    if case["step"]:
        for t in state["inputs"]:
            t.requires_grad_()
    return state


def _forward(state):
    case, inputs = state["case"], state["inputs"]
    op = case["op"]
    if op in BLOCKS:
        return state["block"](inputs[0], *state["extra"])
    if op == "linear":
        return linear_attention(*inputs)
    if op == "simple":
        return simple_la(*inputs)
    if op == "decoupled":
        return decoupled_la(*inputs)
    if op == "varlen":
        return varlen_linear_attention(*inputs, state["cu"], state["longest"])
    return piecewise_sparse_attention(*inputs, density=case["density"], block_size=case["block"])


def run(state):
    if not state["case"]["step"]:
        with torch.no_grad():
            return _forward(state)
    leaves = list(state["inputs"])
    if "block" in state:
        leaves += list(state["block"].parameters())
    for t in leaves:
        t.grad = None
    out = _forward(state)
    out.backward(state["grad"])
    return [out.detach()] + [t.grad for t in leaves]


def _operator_work(rows, keys, DK, DV, size, step, extra=0):
    """Bytes and operations of softmax-free attention over `rows` (token, head) pairs with `keys` of keys and values;
    `extra`: how many more tensors of features each side has (the decoupled operator's plain rows)."""
    q, k, v, o = rows * DK * (1 + extra), keys * DK * (1 + extra), keys * DV, rows * DV
    forward, flops = q + k + v + o, 2 * (rows + keys) * DK * DV
    # backward: q, k, v and the output's gradient in, three gradients out; dS, dq from the rows, dk, dv from the keys
    moved = forward + (q + k + v + o) + (q + k + v) if step else forward
    return {"bytes": moved * size, "flops": flops + (4 * (rows + keys) * DK * DV if step else 0)}


def work(case):
    size, step, op = BYTES[case["dtype"]], case["step"], case["op"]
    if op == "varlen":
        rows = int(_lengths(case).sum()) * case["H"]
        return _operator_work(rows, rows, case["DK"], case["DV"], size, step)
    if op in DENSE:
        rows = case["B"] * case["H"] * case["T"]
        return _operator_work(rows, rows, case["DK"], case["DV"], size, step, extra=int(op == "decoupled"))
    if op == "piecewise":
        rows, D = case["B"] * case["H"] * case["T"], case["DK"]
        blocks = -(-case["T"] // case["block"])
        chosen = max(1, int(case["density"] * blocks))
        pairs = rows * (chosen * case["block"] + (blocks - chosen))
        return {"bytes": 4 * rows * D * size, "flops": 4 * pairs * D + 4 * rows * D * D}
    # blocks: the input and the output (training: the output's gradient in, the input's out as well) and the weights
    # (training: read twice, their gradients written); the projections, the depth-wise convolution and the operator
    tokens, dim, heads = case["B"] * case["side"] ** 2, case["dim"], case["heads"]
    keys, d = tokens // case["sr"] ** 2, dim // case["heads"]
    if op == "linfusion":
        dense, taps, DK, DV = 8 * tokens * dim * dim, 0, d, d
    elif op == "mlla":
        dense, taps, DK, DV = 2 * tokens * dim * dim, 9, d, d
    elif op == "rala":
        dense, taps, DK, DV = 5 * tokens * dim * dim, 25, d, d
    else:
        dense = (2 if op == "focused" else 3) * tokens * dim * dim + 2 * keys * dim * dim
        dense += tokens * dim * dim if case["sr"] > 1 else 0
        taps, DK, DV = 25, (d if op == "focused" else 2 * d), d
    weights = sum(p.numel() for p in _block(case).parameters())
    attention = _operator_work(tokens * heads, keys * heads, DK, DV, size, step)["flops"]
    flops = (2 * dense + 2 * taps * tokens * dim) * (3 if step else 1) + attention
    return {"bytes": ((4 if step else 2) * tokens * dim + (3 if step else 1) * weights) * size, "flops": flops}


def tolerance(case):
    """About four times what a pass was measured to be from its own formula in 64 bits on the same inputs: the
    operators 1.1e-6 (fp32), 2.9e-4 (fp16) and 1.7e-3 (bf16, piecewise attention 2.3e-3); the blocks 9e-6 (fp32, the
    weights of the convolution), 2.2e-3 (fp16) and 1.7e-2 (bf16, the polarity power)."""
    if case["op"] in BLOCKS:
        return {"rel": {"fp32": 4e-5, "fp16": 9e-3, "bf16": 3e-2}[case["dtype"]]}
    if case["op"] == "piecewise":
        return {"rel": {"fp16": 1.2e-3, "bf16": 9e-3}[case["dtype"]]}
    return {"rel": {"fp32": 5e-6, "fp16": 1.2e-3, "bf16": 7e-3}[case["dtype"]]}
