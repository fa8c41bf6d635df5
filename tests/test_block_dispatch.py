"""What the blocks' fused steps take and what they leave to the torch compositions, decided on the host: nothing here
launches a kernel.  A call that torch's operators refuse stays refused, one that they run stays theirs."""
import os
import subprocess
import sys
import threading
import time

import pytest
import torch
import torch.fx
import torch.nn as nn
from torch.autograd import forward_ad
from torch.utils.flop_counter import FlopCounterMode

from flash_bla import _hip
from flash_bla.layers import (FocusedLinearAttention, GeneralizedLinearAttention, MambaLikeLinearAttention,
                              PolaLinearAttention, RALALinearAttention)
from flash_bla.layers import _features as features
from flash_bla.layers import _whole
from flash_bla.layers import focused_la, linfusion, mlla, polaformer, rala
from flash_bla.layers._common import torch_linear_attention
from flash_bla.layers.mlla import RoPE
from flash_bla.ops import depthwise, projection
from flash_bla.ops._check import untouched


@pytest.mark.parametrize("H,W", [(5, 4), (4, 3), (8, 8), (2, 2), (16, 2)])
def test_token_convolution_refuses_a_grid_that_is_not_the_tokens(H, W, monkeypatch):
    """16 tokens: the reshape of the torch composition raises, and no kernel sees the call."""
    monkeypatch.setattr(depthwise, "runs_on_tokens", lambda *a: True)
    monkeypatch.setattr(depthwise.DepthwiseConvTokensFunction, "apply", lambda *a: pytest.fail("reached the kernel"))
    conv, x = nn.Conv2d(8, 8, 3, padding=1, groups=8), torch.randn(2, 16, 16)
    with pytest.raises(RuntimeError):
        depthwise.depthwise_conv_tokens(x, conv, H, W)
    with pytest.raises(ValueError, match="H \\* W"):
        _hip.dwconv_fwd(x, conv.weight, conv.bias, H, W)
    with pytest.raises(ValueError, match="H \\* W"):
        _hip.dwconv_grad(x, x, conv.weight, H, W, True)
    with pytest.raises(ValueError, match="one shape"):
        _hip.dwconv_grad(x, x[:, :-1], conv.weight, 4, 4, True)


def test_token_convolution_entry_point_refuses_overlapping_output_batches():
    L, at = _hip.lib(), 4096  # an aligned address that is never looked at
    args = (at, 16 * 8, 8, at, None, at)
    for y_batch, y_row in ((8 * 15, 8), (8, 8), (16, 8)):
        assert L.fbla_dwconv_fwd(*args, y_batch, y_row, 2, 4, 4, 8, 8, 3, 0, _hip.F16, None) == -1
        assert b"overlap" in L.fbla_last_error()


@pytest.mark.parametrize("dims", [(100, 100), (65, 9), (9, 121)])
def test_ragged_heads_without_the_one_kernel_pass_a_keep_the_widened_copies(dims):
    """More packed heads than that kernel addresses: the two kernels that replace it read rows of whole pieces, so the
    workspace grows with the tokens by widened copies of q, k, v, dO and of the gradients; one head fewer: in place, it
    does not grow.  (One side is 64 wide or more throughout.)"""
    L, (DK, DV), T = _hip.lib(), dims, 64

    def growth(H):
        need = [L.fbla_varlen_workspace_bytes(1, t, 2, H, 32, DK, DV, _hip.BF16, _hip.NORMALIZE) for t in (T, 2 * T)]
        return need[1] - need[0]
    assert growth(65537) >= 2 * T * 65537 * (4 * ((DK + 7) // 8 * 8) + 3 * ((DV + 7) // 8 * 8))
    assert growth(65536) == 0


@pytest.mark.parametrize("L,DK,DV", [(257, 8, 13), (257, 8, 60), (4093, 100, 100), (1000, 66, 9)])
def test_backward_workspace_of_ragged_heads_holds_the_generic_kernels(L, DK, DV):
    """They take over while single phases are timed: one state partial and mean key per chunk of 64 tokens (the shortest
    chunk, taken by a single head of up to 65536 tokens), S^T, s dS, (s dS)^T, dkm, each rounded up to 256 bytes."""
    up = lambda n: (n + 255) // 256 * 256  # noqa: E731
    need = up((L + 63) // 64 * (DK * DV + DK) * 4) + 3 * up(DK * DV * 4) + up(DK * 4)
    for dtype in (_hip.F16, _hip.BF16):
        assert _hip.lib().fbla_la_workspace_bytes(1, 1, 1, L, DK, DV, dtype, _hip.NORMALIZE) >= need


def test_forward_workspace_of_ragged_heads_holds_the_generic_kernels():
    """The same with three times as many keys as queries, where the partials outgrow the widened copies: chunks of 64
    keys."""
    up = lambda n: (n + 255) // 256 * 256  # noqa: E731
    need = _hip.lib().fbla_la_cross_workspace_bytes(0, 1, 1, 1000, 3000, 127, 126, _hip.BF16, _hip.NORMALIZE)
    assert need >= up((3000 + 63) // 64 * (127 * 126 + 127) * 4)


@pytest.mark.parametrize("H,L,D", [(1, 8192, 64), (1, 4096, 128), (3, 4096, 64), (2, 4096, 128), (16, 512, 64)])
def test_long_heads_are_not_cut_finer_than_their_partials_are_worth(H, L, D):
    """The forward's workspace holds one state partial a chunk: few heads are cut until 32 workgroups run, no further."""
    slot = (D * D + D) * 4
    need = _hip.lib().fbla_la_workspace_bytes(0, 1, H, L, D, D, _hip.F16, _hip.NORMALIZE)
    assert need <= max(32, H * L // 256) * slot + 4096


@pytest.mark.parametrize("H", [1, 4, 16])
def test_short_16_bit_heads_keep_two_chunks(H):
    """Up to 512 tokens of 64 x 64: two state partials a head (fp32: more)."""
    slot = 4 * (64 * 64 + 64)
    need = [_hip.lib().fbla_la_workspace_bytes(0, 1, H, 512, 64, 64, dtype, _hip.NORMALIZE) // slot for dtype in (_hip.BF16, _hip.F32)]
    assert need[0] == 2 * H < need[1]


@pytest.mark.parametrize("B,H,L,DK,DV,dtype,flags", [
    (3, 3, 1750, 110, 87, _hip.F16, 0), (4, 1, 1704, 126, 126, _hip.F32, 1), (8, 2, 648, 83, 114, _hip.BF16, 3),
    (1, 16, 689, 76, 123, _hip.F16, 3), (2, 2, 3520, 121, 84, _hip.BF16, 0), (7, 1, 1140, 125, 97, _hip.F32, 1)])
def test_finer_chunks_do_not_take_a_forward_past_the_built_in_scratch(B, H, L, DK, DV, dtype, flags):
    """fbla_la_fwd_static took these: their chunks of 256 tokens need less than the scratch, finer ones more."""
    need = _hip.lib().fbla_la_workspace_bytes(0, B, H, L, DK, DV, dtype, flags)
    assert need <= _hip.lib().fbla_static_scratch_bytes()


@pytest.mark.parametrize("dtype,K,workgroups", [(_hip.F32, 3, 1024), (_hip.F32, 5, 1024), (_hip.F32, 7, 1024), (_hip.BF16, 7, 1024),
                                                (_hip.F16, 7, 1024), (_hip.BF16, 5, 768), (_hip.F16, 3, 768)])
def test_filter_gradients_fill_the_gpu_with_what_their_registers_allow(dtype, K, workgroups):
    """One partial of K * (K + 1) sums a chunk; K tap rows and 4 blocks of channels share the workgroups."""
    need = _hip.lib().fbla_dwconv_grad_workspace_bytes(64, 28, 28, 256, 32, K, dtype)
    assert need == 4 * (workgroups // (4 * K)) * K * (K + 1) * 256


class _Described(torch.Tensor):
    is_cuda = True


def _on_gpu(x):
    """x with the properties of a GPU tensor, for rules that look at no more than those."""
    return x.as_subclass(_Described)


@pytest.mark.parametrize("types", [(torch.bfloat16, torch.float32), (torch.float32, torch.float16), None])
def test_token_convolution_leaves_a_bias_of_another_type_to_torch(types, monkeypatch):
    """nn.Conv2d refuses it; the kernel would read its bytes as x's type."""
    monkeypatch.setattr(depthwise, "plain_tensors", lambda *a: True)
    for bias in (True, False):
        conv = nn.Conv2d(8, 8, 3, padding=1, groups=8, bias=bias)
        x = _on_gpu(torch.randn(2, 16, 16))
        assert depthwise.runs_on_tokens(x, conv)
        if types:
            conv, x = conv.to(types[0]), _on_gpu(x.to(types[0]))
            assert depthwise.runs_on_tokens(x, conv)
        if bias:
            conv.bias = nn.Parameter(conv.bias.detach().to(types[1]) if types else torch.zeros(8, device="meta"))
            assert not depthwise.runs_on_tokens(x, conv)
    for w, b in ((torch.half, torch.float), (torch.float, torch.half)):
        with pytest.raises(ValueError, match="dtype"):
            _hip.dwconv_fwd(torch.randn(2, 16, 16).to(w), torch.randn(8, 1, 3, 3).to(w), torch.zeros(8, dtype=b), 4, 4)


@pytest.mark.parametrize("make", [lambda: nn.Conv2d(8, 8, 3, padding=1, groups=8), lambda: RoPE((4, 4, 8))])
def test_modules_that_do_more_than_their_class_are_not_stood_in_for(make):
    module = make()
    kind, nothing = type(module), lambda *a: None
    assert untouched(module, kind) and not untouched(module, nn.Module)
    for register in (module.register_forward_hook, module.register_forward_pre_hook, module.register_full_backward_hook,
                     module.register_full_backward_pre_hook, nn.modules.module.register_module_forward_hook,
                     nn.modules.module.register_module_forward_pre_hook,
                     nn.modules.module.register_module_full_backward_hook,
                     nn.modules.module.register_module_full_backward_pre_hook):
        hook = register(nothing)
        assert not untouched(module, kind)
        hook.remove()
        assert untouched(module, kind)
    module.forward = nothing
    assert not untouched(module, kind)
    del module.forward
    module.compile(backend="eager")
    assert not untouched(module, kind)


BLOCKS = {
    "linfusion": (lambda: GeneralizedLinearAttention(16, heads=2, dim_head=8), ()),
    "mlla": (lambda: MambaLikeLinearAttention(16, (4, 4), 2), ()),
    "rala": (lambda: RALALinearAttention(16, (4, 4), 2), ()),
    "focused": (lambda: FocusedLinearAttention(16, 16, num_heads=2, sr_ratio=2), (4, 4)),
    "pola": (lambda: PolaLinearAttention(16, 16, num_heads=2), (4, 4)),
}


@pytest.mark.parametrize("name", sorted(BLOCKS))
def test_blocks_hold_plain_linear_modules_and_project_through_the_kernel_function(name, monkeypatch):
    """By type they are nn.Linear, every one of them is offered to the token-splitting function, and one that is hooked or
    replaced runs as the module that it is."""
    make, extra = BLOCKS[name]
    block, x = make(), torch.randn(2, 16, 16)
    layers = [m for m in block.modules() if isinstance(m, nn.Linear)]
    assert len(layers) >= 1 and all(type(m) is nn.Linear for m in layers)
    want = block(x, *extra, mode="torch")

    weights = []
    monkeypatch.setattr(projection, "runs_on_rows", lambda x, weight, bias: True)
    monkeypatch.setattr(projection.TokenLinearFunction, "apply",
                        lambda x, weight, bias: weights.append(weight) or nn.functional.linear(x, weight, bias))
    assert torch.equal(block(x, *extra, mode="torch"), want)
    assert {id(w) for w in weights} == {id(m.weight) for m in layers}

    seen = []
    for m in layers:
        m.register_forward_hook(lambda m, args, out: seen.append(m))
    del weights[:]
    assert torch.equal(block(x, *extra, mode="torch"), want) and not weights
    assert {id(m) for m in seen} == {id(m) for m in layers}


FUSED = (features.PolarityFeaturesFunction, features.FocusedFeaturesFunction, features.RotaryFeaturesFunction,
         features.TurnedHeadsFunction, features.MergeHeadsFunction, features.InterpolateTokensFunction)


@pytest.fixture
def only_shapes_decide(monkeypatch):
    """Every tensor counts as one that the kernels could read; a call that reaches them is reported."""
    class Reached(Exception):
        pass

    def reached(*args):
        raise Reached
    monkeypatch.setattr(features, "_takes", lambda *a: True)
    monkeypatch.setattr(features, "elu_plus_one", lambda t: nn.functional.elu(t) + 1)
    for function in FUSED:
        monkeypatch.setattr(function, "apply", reached)
    return Reached


# 2 batches of 9 queries and 4 keys, 2 heads of 8 channels
ROWS, KEYS, HEADS, DIM = 9, 4, 2, 16


def _features_call(name, **shapes):
    t = {k: torch.rand(v) for k, v in shapes.items()}
    if name == "polarity":
        args = (t["qg"], t["kv"], t["pe"], t["scale"], t["power"], HEADS)
        return features.polarity_features(*args), features.polarity_formula(*args)
    if name == "focused":
        args = (t["q"], t["kv"], t["pe"], t["scale"], HEADS, 3)
        return features.focused_features(*args), features.focus_formula(*args)
    if name == "rotary":
        args = (t["qk"], t["x"], t["rotations"], 3, HEADS)
        return features.rotary_features(*args), features.rotary_formula(*args)
    args = t["o"], t.get("o2"), t["local"], t.get("gate")
    return (features.merge_heads_with(*args),), features.merge_formula(*args)


FULL = {
    "polarity": dict(qg=(2, ROWS, 2 * DIM), kv=(2, KEYS, 2 * DIM), pe=(1, KEYS, DIM), scale=(1, 1, DIM),
                     power=(1, HEADS, 1, DIM // HEADS)),
    "focused": dict(q=(2, ROWS, DIM), kv=(2, KEYS, 2 * DIM), pe=(1, KEYS, DIM), scale=(1, 1, DIM)),
    "rotary": dict(qk=(2, ROWS, 2 * DIM), x=(2, ROWS, DIM), rotations=(3, 3, DIM // 2, 2)),
    "merge": dict(o=(2, HEADS, ROWS, DIM // HEADS), local=(2, ROWS, DIM)),
    "merge halves": dict(o=(2, HEADS, ROWS, DIM // 4), o2=(2, HEADS, ROWS, DIM // 4), local=(2, ROWS, DIM),
                         gate=(2, ROWS, DIM)),
}


@pytest.mark.parametrize("name", sorted(FULL))
def test_full_shapes_reach_the_kernels(name, only_shapes_decide):
    with pytest.raises(only_shapes_decide):
        _features_call(name, **FULL[name])


@pytest.mark.parametrize("name,other", [
    ("polarity", dict(power=(1, 1, 1, 1))), ("polarity", dict(power=(1, 1, 1, DIM // HEADS))),
    ("polarity", dict(power=(1, HEADS, 1, 1))), ("polarity", dict(pe=(1, 1, DIM))), ("polarity", dict(scale=(1, 1, 1))),
    ("polarity", dict(kv=(1, KEYS, 2 * DIM))), ("focused", dict(kv=(1, KEYS, 2 * DIM))), ("focused", dict(scale=(1,))),
    ("focused", dict(pe=(2, KEYS, DIM))), ("merge", dict(local=(1, ROWS, DIM))), ("merge", dict(gate=(1, 1, DIM))),
    ("merge halves", dict(gate=(2, ROWS, 1)))])
def test_shapes_that_torch_broadcasts_run_as_torch_operators(name, other, only_shapes_decide):
    """A replaced parameter of fewer elements: the kernels would read past it."""
    got, want = _features_call(name, **{**FULL[name], **other})
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("name,other", [
    ("polarity", dict(power=(1, HEADS, ROWS, DIM))), ("polarity", dict(kv=(2, KEYS, 2 * DIM + 16))),
    ("focused", dict(kv=(2, KEYS, 4 * DIM))), ("rotary", dict(qk=(2, ROWS, 4 * DIM))), ("rotary", dict(qk=(2, 4, 2 * DIM))),
    ("merge", dict(local=(2, ROWS - 1, DIM))), ("merge", dict(gate=(2, ROWS, DIM // 2))),
    ("merge halves", dict(o2=(2, HEADS, ROWS - 1, DIM // 4)))])
def test_shapes_that_torch_refuses_stay_refused(name, other, only_shapes_decide):
    with pytest.raises(RuntimeError):
        _features_call(name, **{**FULL[name], **other})


@pytest.mark.parametrize("name", sorted(BLOCKS))
def test_blocks_in_torch_mode_can_be_traced(name):
    """torch.jit.trace of a block that trains, and torch.fx where the block's own code allows it, see the projections as the
    modules that they are."""
    make, extra = BLOCKS[name]
    block, x = make(), torch.randn(2, 16, 16)

    class TorchMode(nn.Module):
        def __init__(self):
            super().__init__()
            self.block = block

        def forward(self, x):
            return self.block(x, *extra, mode="torch")
    layers = {n for n, m in block.named_modules() if type(m) is nn.Linear}
    traced = torch.jit.trace(TorchMode(), x)
    torch.testing.assert_close(traced(x), block(x, *extra, mode="torch"))
    assert {n for n in layers if n.count(".") == 0} <= {n.removeprefix("block.") for n, _ in traced.named_modules()}
    if name not in ("mlla", "rala"):  # (int() of the number of tokens)
        fixed = {"H": 4, "W": 4} if extra else {"encoder_hidden_states": None, "attention_mask": None}
        graph = torch.fx.symbolic_trace(block, concrete_args={"mode": "torch", **fixed}).graph
        assert layers <= {n.target for n in graph.nodes if n.op == "call_module"}


def test_traced_and_watched_calls_are_not_plain():
    x = torch.randn(2, 3)
    seen = []
    torch.jit.trace(lambda t: seen.append(projection.plain_tensors(t)) or t + 1, x, check_trace=False)
    assert projection.plain_tensors(x) and seen and not any(seen)
    with FlopCounterMode(display=False):
        assert not projection.plain_tensors(x)


def _cpu_kernels(monkeypatch):
    """The forward kernels by their formulas; a gradient kernel asks for its tensors' addresses and fails the test."""
    n = features

    def read(*args):
        addresses = [t.data_ptr() for t in args if torch.is_tensor(t)]
        pytest.fail(f"a kernel read what it cannot: {addresses}")
    for name, formula in (("polarity_fwd", lambda *a: n.polarity_formula(*a)[:4]), ("focus_fwd", lambda *a: n.focus_formula(*a)[:3]),
                          ("rotary_fwd", lambda qk, x, rot, heads: n.rotary_formula(qk, x, rot, rot.shape[0], heads)[:5]),
                          ("turn_fwd", n.turn_formula), ("merge_fwd", lambda *a: n.merge_formula(*a)[0]),
                          ("interpolate_fwd", lambda *a: n.interpolate_formula(*a)[0]),
                          ("dwconv_fwd", lambda x, w, b, H, W, flip=False: read(x) if flip else _conv_formula(x, w, b, H, W))):
        monkeypatch.setattr(_hip, name, formula)
    for name in ("polarity_bwd", "focus_bwd", "rotary_bwd", "turn_bwd", "merge_bwd", "interpolate_bwd", "dwconv_grad",
                 "linear_wgrad"):
        monkeypatch.setattr(_hip, name, read)


def _conv_formula(x, w, b, H, W):
    return depthwise._convolution_of_images(x, H, W, w.shape[0], lambda i: nn.functional.conv2d(
        i, w, b, padding=1, groups=w.shape[0]))


_ANGLES = torch.arange(9 * 8.0).reshape(3, 3, 8)
ROTATIONS = torch.stack([_ANGLES.cos(), _ANGLES.sin()], dim=-1)
NODES = {  # function, the same by torch's operators, shapes of the inputs, what follows them
    "polarity": (features.PolarityFeaturesFunction, features.polarity_formula, tuple(FULL["polarity"].values()), (HEADS,)),
    "focused": (features.FocusedFeaturesFunction, features.focus_formula, tuple(FULL["focused"].values()), (HEADS,)),
    "rotary": (features.RotaryFeaturesFunction, features.rotary_formula, tuple(FULL["rotary"].values())[:2],
               (ROTATIONS, 3, HEADS)),
    "turned": (features.TurnedHeadsFunction, features.turn_formula, ((2, HEADS, 9, 8),) * 2 + ((2, HEADS, 9, 1),),
               (ROTATIONS[:, :, :4].contiguous(),)),
    "merge": (features.MergeHeadsFunction, lambda o, local, *rest: features.merge_formula(o, None, local, None),
              tuple(FULL["merge"].values()), ()),
    "merge halves": (features.MergeHeadsFunction, features.merge_formula, tuple(FULL["merge halves"].values()), ()),
    "interpolate": (features.InterpolateTokensFunction, features.interpolate_formula, ((2, 4, 8),), (9,)),
    "convolution": (depthwise.DepthwiseConvTokensFunction, _conv_formula, ((2, 9, 16), (8, 1, 3, 3), (8,)), (3, 3)),
    "projection": (projection.TokenLinearFunction, nn.functional.linear, ((2, 9, 16), (24, 16), (24,)), ()),
}


@pytest.mark.parametrize("how", ["batches", "tangents", "mapped", "twice"])
@pytest.mark.parametrize("name", sorted(NODES))
def test_gradients_that_kernels_cannot_read_are_composed(name, how, monkeypatch):
    """Batches of gradients (is_grads_batched), gradients that carry tangents, gradients inside torch.func.vmap and
    gradients of gradients give what torch's operators give."""
    _cpu_kernels(monkeypatch)
    function, formula, shapes, rest = NODES[name]
    torch.manual_seed(0)
    inputs = [(torch.rand(s) + 0.5).requires_grad_() for s in shapes]
    if name == "merge":
        out = function.apply(inputs[0], None, inputs[1], None)
    else:
        out = function.apply(*inputs, *rest)
    results = []
    for o in (out, formula(*inputs, *rest)):
        o = (o,) if torch.is_tensor(o) else tuple(o)
        gen = torch.Generator().manual_seed(1)
        g, t = ([torch.randn(3, *x.shape, generator=gen) for x in o] for _ in range(2))
        if how == "batches":
            got = torch.autograd.grad(o, inputs, g, is_grads_batched=True)
        elif how == "mapped":
            got = torch.func.vmap(lambda *g: torch.autograd.grad(o, inputs, g, retain_graph=True))(*g)
        elif how == "tangents":
            with forward_ad.dual_level():
                dual = [forward_ad.make_dual(a[0], b[0]) for a, b in zip(g, t)]
                got = [x for d in torch.autograd.grad(o, inputs, dual) for x in forward_ad.unpack_dual(d)]
        else:
            first = torch.autograd.grad(o, inputs, [a[0] for a in g], create_graph=True)
            got = torch.autograd.grad(sum(x.square().sum() for x in first if x.requires_grad), inputs, allow_unused=True) \
                if any(x.requires_grad for x in first) else []
        results.append([x for x in got if x is not None])
    assert len(results[0]) == len(results[1])
    for a, b in zip(*results):
        assert not a.requires_grad
        # fp32 sums of at most 36 products in another order; NaN: the power's second derivative at 0
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4, equal_nan=True)


@pytest.mark.parametrize("alpha,fused", [(4, True), (0.0, True), (-0.5, False), (torch.tensor(4.0), False)])
def test_powers_below_one_run_as_torch_operators(alpha, fused, monkeypatch):
    """0 to a power below 1 has an infinite slope: the kernels take the gradient there for zero, as it is from 1 on."""
    class Reached(Exception):
        pass

    def reached(*args):
        raise Reached
    monkeypatch.setattr(polaformer, "polarity_features" if fused else "polarity_formula", reached)
    block = PolaLinearAttention(16, 16, num_heads=2, alpha=alpha)
    with pytest.raises(Reached):
        block(torch.randn(2, 16, 16), 4, 4)


@pytest.mark.parametrize("side,dtype,fused", [(16, torch.half, True), (256, torch.half, False), (256, torch.bfloat16, True)])
def test_rala_scores_times_tokens_that_overflow_are_not_formed(side, dtype, fused, monkeypatch):
    """65536 tokens in fp16: a score of 1 times n is infinite, and a key of 0 times that is NaN; (k * score) * n is not."""
    class Reached(Exception):
        pass

    def reached(*args):
        raise Reached
    monkeypatch.setattr(rala, "turned_heads", reached)
    block = RALALinearAttention(8, (side, side), 1).to(dtype)
    block.rope.float()
    with pytest.raises(Reached if fused else ValueError, match=None if fused else "GPU"), torch.no_grad():
        block(torch.zeros(1, side * side, 8, dtype=dtype))


@pytest.mark.parametrize("factor", [2.5, nn.Parameter(torch.tensor(3.0)), torch.tensor(3.0)])
def test_focusing_factors_that_are_not_the_number_three_run_as_torch_operators(factor, only_shapes_decide):
    """A learned factor of exactly 3 has a gradient, which the cube's kernel does not give."""
    q, kv, pe, scale = (torch.rand(s) + 0.5 for s in FULL["focused"].values())
    out = features.focused_features(q, kv, pe, scale, HEADS, factor)
    for a, b in zip(out, features.focus_formula(q, kv, pe, scale, HEADS, factor)):
        assert torch.equal(a, b)
    if isinstance(factor, nn.Parameter):
        assert torch.autograd.grad(out[0].sum(), factor)[0] != 0
    with pytest.raises(only_shapes_decide):
        features.focused_features(q, kv, pe, scale, HEADS, 3.0)


def test_composed_gradients_stop_at_their_inputs():
    """One input made of another: the gradient of the step is composed without walking from one to the other (whose
    nodes would run twice)."""
    seen = []
    a = torch.rand(2, HEADS, ROWS, 8, requires_grad=True)
    o = a * 1
    o.register_hook(lambda g: seen.append(1))
    local = torch.rand(2, ROWS, DIM, requires_grad=True)
    gate = (o * 2).transpose(1, 2).reshape(2, ROWS, DIM)
    grads = features.differentiable_gradients(features.merge_formula, (o, None, local, gate), (torch.ones(2, ROWS, DIM),))
    assert not seen and [g is None for g in grads] == [False, True, False, False]
    assert torch.equal(grads[0], features.split_heads(gate, HEADS).detach())


@pytest.fixture
def native(monkeypatch):
    """Blocks that run whole on the CPU: every call fits; the native calls note the numbers they are given and return zeros."""
    seen = []

    def numbers(args):
        return [a for a in args if type(a) in (int, float)]

    def forward(x, *args):
        seen.append(numbers(args))
        return [torch.zeros_like(x), x.detach()]

    def backward(g, x, *args):
        seen.append(numbers(args))
        need = next(a for a in args if isinstance(a, (list, tuple)) and all(type(e) is bool for e in a))
        return [torch.zeros_like(x)] + [None] * (len(need) - 1)
    monkeypatch.setattr(_whole, "_ordinary", lambda *a: True)
    monkeypatch.setattr(_hip, "plain_gpu_tensors", lambda *a: True)
    for name in ("mlla", "pola", "focused", "linfusion"):
        monkeypatch.setattr(_hip, name + "_fits", lambda *a: True)
        monkeypatch.setattr(_hip, name + "_fwd", forward)
        monkeypatch.setattr(_hip, name + "_bwd", backward)
    return seen


@pytest.mark.parametrize("name", ["mlla", "pola", "focused"])
def test_numbers_of_a_whole_call_are_those_of_its_forward(name, native):
    """A schedule moves them, two calls of different numbers share a backward: each has its own."""
    make, extra = BLOCKS[name]
    block, x = make(), torch.randn(2, 16, 16, requires_grad=True)
    out = [block(x, *extra)]
    block.alpha, block.num_heads = 1.5, 4
    out.append(block(x, *extra))
    block.alpha, block.num_heads = 2.5, 1
    (out[0] + out[1]).sum().backward()
    assert len(native) == 4 and native[0] != native[1] and sorted(native[2:]) == sorted(native[:2])


def test_a_whole_call_saves_what_its_backward_reads(native):
    """A rotation that is written between forward and backward is noticed, and saved-tensor hooks see it."""
    make, extra = BLOCKS["mlla"]
    block, x, packed = make(), torch.randn(2, 16, 16, requires_grad=True), []
    out = block(x, *extra)
    with torch.no_grad():
        block.rope.rotations.mul_(2)
    with pytest.raises(RuntimeError, match="inplace"):
        out.sum().backward()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
        block(x, *extra)
    assert any(t is block.rope.rotations or t.data_ptr() == block.rope.rotations.data_ptr() for t in packed)


@pytest.fixture
def torch_operators(monkeypatch):
    """The attention operators by torch's on the CPU."""
    def paired(q1, q2, k, v):
        return tuple(torch_linear_attention(q, k, part) for q, part in zip((q1, q2), v.chunk(2, dim=-1)))

    def packed(q, k, v, cu, n, eps, feature_map):
        heads = [t.unflatten(0, (-1, n)).transpose(1, 2) for t in (nn.functional.elu(q) + 1, nn.functional.elu(k) + 1, v)]
        return torch_linear_attention(*heads, eps=eps).transpose(1, 2).flatten(0, 1)
    for module in (mlla, features):
        monkeypatch.setattr(module, "elu_plus_one", lambda t: nn.functional.elu(t) + 1)
    monkeypatch.setattr(mlla, "decoupled_la", lambda q, k, q_rope, k_rope, v, scale: torch_linear_attention(
        q, k, v, q_num=q_rope, k_num=k_rope))
    monkeypatch.setattr(polaformer, "paired_linear_attention", paired)
    monkeypatch.setattr(focused_la, "linear_attention", torch_linear_attention)
    monkeypatch.setattr(linfusion, "varlen_linear_attention", packed)


@pytest.mark.parametrize("name", ["mlla", "pola", "focused", "linfusion"])
def test_composed_gradients_of_a_whole_call_are_those_of_its_forward(name, native, torch_operators, monkeypatch):
    """Gradients of gradients, of parameters that two projections share, after the module has got other numbers, hooks and
    parameters; the module is not touched meanwhile."""
    make, extra = BLOCKS[name]
    torch.manual_seed(0)
    block, x, g = make(), torch.randn(2, 16, 16, requires_grad=True), torch.randn(2, 16, 16)
    with torch.no_grad():
        for p in block.parameters():
            p.add_(0.1 * torch.randn(p.shape))
    if name == "linfusion":
        block.to_k.weight = block.to_q.weight
        block.to_q_[2].negative_slope = 0.3
    elif name == "pola":
        block.qg.weight = block.kv.weight
    elif name == "focused":
        block.proj.weight = block.q.weight
    wanted = [x, *(p for n, p in block.named_parameters() if not n.startswith(("sr", "norm")))]

    def gradients(out):
        once = torch.autograd.grad(out, wanted, g, create_graph=True)
        return once, torch.autograd.grad(sum(t.square().sum() for t in once), wanted, allow_unused=True)
    want = gradients(block(x, *extra, mode="torch"))
    if name == "linfusion":
        call = _whole._LinFusion(block, GeneralizedLinearAttention)
        paths, rest = (block.to_q_, block.to_k_), (block.to_q, block.to_k, block.to_v, block.to_out[0])
        params = [t for p in paths for i in (0, 1, 3) for t in (p[i].weight, p[i].bias)] + [t for m in rest for t in (m.weight, m.bias)]
        monkeypatch.setattr(_hip, "linfusion_fwd", lambda x, *a: [torch.zeros_like(x)])
        out = _whole.WholeBlockFunction.apply(call, x, *params, torch.tensor([0, 16, 32], dtype=torch.int32))
        block.to_q_[2].negative_slope = block.to_k_[1].eps = 0.7
        block.heads = 1
    else:
        out = block(x, *extra)
        block.num_heads, block.alpha, block.focusing_factor = 1, 0.5, 1
    for m in list(block.modules())[1:]:
        m.register_forward_hook(lambda m, args, out: pytest.fail("the module ran"))
    for m in block.children():
        m.weight = nn.Parameter(torch.zeros(3))
    for got, expected in zip(gradients(out), want):
        assert [t is None for t in got] == [t is None for t in expected]
        for a, b in zip(got, expected):
            if a is not None:  # fp32 sums of at most 64 products in another order; NaN: the power's second derivative at 0
                torch.testing.assert_close(a, b, rtol=1e-3, atol=1e-4 * float(b.detach().nan_to_num().abs().max() + 1), equal_nan=True)


@pytest.mark.parametrize("slope,kept", [(0.01, True), (0, True), (-0.1, False), (float("nan"), False), (torch.tensor(0.1), False)])
def test_slopes_that_turn_signs_run_step_by_step(slope, kept):
    assert _whole._keeps_signs(nn.LeakyReLU(slope)) == kept


def test_function_modes_are_noticed():
    """What watches or replaces torch's functions sees a block's steps; a default device is no such thing."""
    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    assert not _whole._watched()
    with torch.device("cpu"):
        assert not _whole._watched()
        with Watch():
            assert _whole._watched()
        assert not _whole._watched()


def test_layers_import_where_a_private_name_of_functorch_is_missing():
    """A torch without it has every layer; only gradients inside torch.func.vmap ask for it."""
    code = ("import torch, torch._functorch.pyfunctorch as p; del p.temporarily_clear_interpreter_stack; "
            "import flash_bla.layers")
    path = os.pathsep.join(p for p in sys.path if p)
    subprocess.run([sys.executable, "-c", code], check=True, env={**os.environ, "PYTHONPATH": path})


def test_convolutions_whose_weight_was_replaced_are_not_taken_for_what_they_were():
    """torch reads groups and padding off the module and refuses filters that do not go with them (or leaves a smaller grid)."""
    def conv(**more):
        return nn.Conv2d(8, 8, 3, padding=1, groups=8, **more)
    assert _whole._same_convolution(conv())
    for shape in ((8, 1, 5, 5), (4, 1, 3, 3), (16, 1, 3, 3)):
        other = conv()
        other.weight = nn.Parameter(torch.zeros(shape))
        assert not _whole._same_convolution(other)


@pytest.mark.parametrize("heads", [0, -2])
def test_numbers_of_heads_that_are_none_do_not_fit(heads):
    """Python's division by zero raises, C++'s ends the process."""
    block, x = MambaLikeLinearAttention(64, (4, 4), 2), torch.zeros(1, 16, 64)
    params = (block.qk.weight, block.qk.bias, block.lepe.weight, block.lepe.bias)
    assert _hip.mlla_fits(x, params, block.rope.rotations, 4, 2) and not _hip.mlla_fits(x, params, block.rope.rotations, 4, heads)
    for fits, block, q in ((_hip.pola_fits, PolaLinearAttention(64, 16, num_heads=2, qkv_bias=True), "qg"),
                           (_hip.focused_fits, FocusedLinearAttention(64, 16, num_heads=2, qkv_bias=True), "q")):
        names = [f"{q}.weight", f"{q}.bias", "kv.weight", "kv.bias", "positional_encoding", "scale", "power", "dwc.weight", "dwc.bias",
                 "proj.weight", "proj.bias"]
        named = dict(block.named_parameters())
        params = [named[n] for n in names if n in named]
        assert fits(x, x, params, 4, 4, 2) and not fits(x, x, params, 4, 4, heads)
    rows, heads4 = torch.zeros(1, 16, 128), torch.zeros(1, 2, 16, 32)
    for call in (lambda: _hip.polarity_fwd(rows, rows, rows, rows, rows, heads), lambda: _hip.rotary_fwd(rows, x, rows, heads),
                 lambda: _hip.focus_fwd(x, rows, x, x, heads), lambda: _hip.merge_bwd(x, heads, False, None, None, None, None),
                 lambda: _hip.polarity_bwd(rows, rows, rows, rows, rows, heads, *[rows] * 6),
                 lambda: _hip.rotary_bwd(rows, rows, heads, *[x] * 6), lambda: _hip.focus_bwd(x, rows, x, x, heads, *[x] * 4),
                 lambda: _hip.chunk_reduce(heads4, heads4, heads4, heads), lambda: _hip.norm_leaky([(x[..., :0], None, None, 1e-5, 0.1)], False)):
        with pytest.raises(ValueError, match="positive"):
            call()


def test_native_calls_let_other_threads_run():
    """A call that takes a while (here a projection on the CPU, in front of a kernel that refuses its rows) does not hold the
    interpreter's lock: with a switch interval that no call reaches, the other thread runs only while the lock is given up."""
    x, w = torch.randn(1, 2048, 1024), torch.randn(2048, 1024)
    args = (x, x, [w[:1024], None, w, None, x, x[:, :1], w, None, w, None], 32, 64, 4, False)
    ticks, stop, interval = [0], threading.Event(), sys.getswitchinterval()

    def tick():
        while not stop.is_set():
            ticks[0] += 1
            time.sleep(0)
    thread = threading.Thread(target=tick)
    thread.start()
    try:
        sys.setswitchinterval(1000)
        before = ticks[0]
        with pytest.raises(ValueError, match="GPU"):
            _hip.focused_fwd(*args)
        during = ticks[0] - before
    finally:
        stop.set()
        sys.setswitchinterval(interval)
        thread.join()
    assert during > 0


@pytest.mark.parametrize("tokens,K,N,alone,several", [
    (50176, 256, 256, False, True), (50176, 128, 256, False, True), (12544, 512, 512, False, True), (12544, 256, 512, False, True),
    (50176, 256, 512, True, True), (12544, 256, 256, True, True), (8192, 640, 640, True, True), (200704, 64, 128, True, True),
    (4096, 1280, 1280, False, False), (12544, 512, 1024, False, False), (64, 64, 65544, False, False), (8, 40000, 20000, False, False)])
def test_products_that_the_library_is_faster_at_are_left_to_it(tokens, K, N, alone, several):
    """Large ones of whole tiles, by themselves; and what the kernel's entry point refuses."""
    x, w = torch.empty(tokens, K, dtype=torch.half, device="meta"), torch.empty(N, K, dtype=torch.half, device="meta")
    assert (_hip.projects(x, w, True), _hip.projects(x, w, False)) == (alone, several)
    far = torch.empty_strided((4, K), ((1 << 22) + 8, 1), dtype=torch.half, device="meta")
    assert not _hip.projects(far, w, False) and not _hip.projects(x.float(), w.float(), False)
