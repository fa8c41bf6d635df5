"""What the vision blocks do between their projections and the attention operators, one HIP launch a direction: polarity
features (layers/polaformer.py:63-84), focused features (layers/focused_la.py:56-74), rotary features
(layers/mlla.py:74-81), weighted and turned heads (layers/rala.py:60-69), interpolated tokens (focused_la.py:88-91) and
heads merged back to rows (polaformer.py:92-104, mlla.py:88-92).  The reference composes them of torch operators; the
compositions here are what runs when the kernels do not take a call, and what a gradient is made of that is differentiated
again or that the kernels cannot read.
"""
import torch
import torch.nn as nn
import torch.nn.functional as F

from flash_bla import _hip
from flash_bla.layers._common import merge_heads, split_heads
from flash_bla.ops.feature_map import elu_plus_one
from flash_bla.ops.projection import eager_call, gradient_of

_TYPES = (torch.float16, torch.bfloat16, torch.float32)


def _takes(heads, channels, unit, *tensors):
    """Ordinary GPU tensors of one supported type whose heads (or their `unit` parts) are whole 16-byte pieces."""
    x = tensors[0]
    dtype, device = x.dtype, x.get_device()
    if not x.is_cuda or dtype not in _TYPES or channels % heads or channels // heads % (unit * 16 // x.element_size()):
        return False
    for t in tensors:
        if t is not None and (type(t) is not torch.Tensor and type(t) is not nn.Parameter or t.dtype != dtype or
                              t.get_device() != device or not 0 < t.numel() < 1 << 31):
            return False
    return not torch.is_autocast_enabled() and eager_call()


def differentiable_gradients(formula, inputs, grads):
    """Gradients of formula(*inputs) by torch's operators, which can be differentiated again where that is wanted."""
    with torch.enable_grad():
        # (through aliases: the inputs may depend on one another, and the engine would walk from one to the other)
        inputs = [t.view_as(t) if torch.is_tensor(t) and t.requires_grad else t for t in inputs]
        out = formula(*inputs)
    wanted = [t for t in inputs if torch.is_tensor(t) and t.requires_grad]
    pairs = [(o, g) for o, g in zip(out, grads) if o is not None and o.requires_grad]
    got = iter(torch.autograd.grad([o for o, _ in pairs], wanted, [g for _, g in pairs],
                                   create_graph=torch.is_grad_enabled(), allow_unused=True))
    return tuple(next(got) if torch.is_tensor(t) and t.requires_grad else None for t in inputs)


def polarity_formula(qg, kv, pe, scale, power, heads):
    q, gate = qg.chunk(2, dim=-1)
    k, v_rows = kv.chunk(2, dim=-1)
    q, k, v = (split_heads(t, heads) for t in (q / scale, (k + pe) / scale, v_rows))
    q_pos, q_neg, k_pos, k_neg = (F.relu(t) ** power for t in (q, -q, k, -k))
    return (torch.cat([q_pos, q_neg], dim=-1), torch.cat([q_neg, q_pos], dim=-1), torch.cat([k_pos, k_neg], dim=-1), v,
            v_rows, gate)


class PolarityFeaturesFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, qg, kv, pe, scale, power, heads):
        ctx.save_for_backward(qg, kv, pe, scale, power)
        ctx.heads = heads
        return (*_hip.polarity_fwd(qg, kv, pe, scale, power, heads), kv.chunk(2, dim=-1)[1], qg.chunk(2, dim=-1)[1])

    @staticmethod
    def backward(ctx, *grads):
        inputs = (*ctx.saved_tensors, ctx.heads)
        return gradient_of(lambda *g: (*_hip.polarity_bwd(*inputs, *g), None),
                           lambda *g: differentiable_gradients(polarity_formula, inputs, g), *grads)


def polarity_features(qg, kv, pe, scale, power, heads):
    """qg [B, N, 2C] (queries | gate), kv [B, n, 2C] (keys | values), pe [1, n, C], scale [1, 1, C], power [1, heads, 1, d]
    (at least 1).  Returns (q_same, q_opp [B, heads, N, 2d], k_both [B, heads, n, 2d], v [B, heads, n, d], the values as rows
    [B, n, C], the gate [B, N, C])."""
    C = qg.shape[-1] // 2
    if (_takes(heads, C, 1, qg, kv, pe, scale, power) and qg.ndim == 3 and kv.ndim == 3 and qg.shape[2] == 2 * C and
            kv.shape == (qg.shape[0], kv.shape[1], 2 * C) and pe.shape == (1, kv.shape[1], C) and
            scale.shape == (1, 1, C) and power.shape == (1, heads, 1, C // heads)):
        return PolarityFeaturesFunction.apply(qg, kv, pe, scale, power, heads)
    return polarity_formula(qg, kv, pe, scale, power, heads)


def focus(t, scale, factor):
    """relu features sharpened by an element-wise power at constant norm."""
    t = (F.relu(t) + 1e-6) / scale
    norm = t.norm(dim=-1, keepdim=True)
    t = t ** factor
    return t / t.norm(dim=-1, keepdim=True) * norm


def focus_formula(q, kv, pe, scale, heads, factor=3):
    k, v_rows = kv.chunk(2, dim=-1)
    q, k = focus(q, scale, factor), focus(k + pe, scale, factor)
    return (*(split_heads(t, heads) for t in (q, k, v_rows)), v_rows)


class FocusedFeaturesFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, kv, pe, scale, heads):
        ctx.save_for_backward(q, kv, pe, scale)
        ctx.heads = heads
        return (*_hip.focus_fwd(q, kv, pe, scale, heads), kv.chunk(2, dim=-1)[1])

    @staticmethod
    def backward(ctx, *grads):
        inputs = (*ctx.saved_tensors, ctx.heads)
        return gradient_of(lambda *g: (*_hip.focus_bwd(*inputs, *g), None),
                           lambda *g: differentiable_gradients(focus_formula, inputs, g), *grads)


def focused_features(q, kv, pe, scale, heads, factor):
    """q [B, N, C], kv [B, n, 2C] (keys | values), pe [1, n, C], scale [1, 1, C].  Returns (q, k, v [B, heads, tokens, d],
    the values as rows [B, n, C]).  The kernels know the cube (a factor that is a tensor may want a gradient)."""
    C = q.shape[-1]
    if (isinstance(factor, (int, float)) and factor == 3 and _takes(heads, C, 1, q, kv, pe, scale) and
            C <= _hip.most_row_channels(q) and q.ndim == 3 and kv.ndim == 3 and
            kv.shape == (q.shape[0], kv.shape[1], 2 * C) and pe.shape == (1, kv.shape[1], C) and scale.shape == (1, 1, C)):
        return FocusedFeaturesFunction.apply(q, kv, pe, scale, heads)
    return focus_formula(q, kv, pe, scale, heads, factor)


def rotate(x, rotations):
    """Neighbouring channels of x as complex numbers times rotations [..., pairs, 2]; fp32."""
    pairs = torch.view_as_complex(x.float().reshape(*x.shape[:-1], -1, 2))
    return torch.view_as_real(torch.view_as_complex(rotations) * pairs).flatten(-2)


def rotary_formula(qk, x, rotations, side, heads, features=lambda t: F.elu(t) + 1.0):
    b, n, c = x.shape
    q, k = features(qk).chunk(2, dim=-1)
    rot = [rotate(t.reshape(b, side, side, c), rotations).reshape(b, n, c).to(x.dtype) for t in (q, k)]
    return (*(split_heads(t, heads) for t in (q, k, *rot, x)), x)


class RotaryFeaturesFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, qk, x, rotations, side, heads):
        ctx.save_for_backward(qk, x, rotations)
        ctx.side, ctx.heads = side, heads
        return (*_hip.rotary_fwd(qk, x, rotations, heads), x.view_as(x))

    @staticmethod
    def backward(ctx, *grads):
        qk, x, rotations = ctx.saved_tensors
        inputs = qk, x, rotations, ctx.side, ctx.heads
        return gradient_of(lambda *g: (*_hip.rotary_bwd(qk, rotations, ctx.heads, *g), None, None, None),
                           lambda *g: differentiable_gradients(rotary_formula, inputs, g), *grads)


def rotary_features(qk, x, rotations, side, heads):
    """qk [B, N, 2C] (queries | keys before elu + 1), x [B, N, C] (the values), N = side * side, rotations
    [side, side, C / 2, 2].  Returns (q, k, q_rot, k_rot, v [B, heads, N, d], the values as rows)."""
    if (_takes(heads, x.shape[-1], 1, x, qk) and x.ndim == 3 and qk.shape == (*x.shape[:2], 2 * x.shape[2]) and
            type(rotations) is torch.Tensor and rotations.dtype == torch.float32 and
            rotations.device == x.device and not rotations.requires_grad and
            rotations.shape == (side, side, x.shape[2] // 2, 2) and x.shape[1] == side * side):
        return RotaryFeaturesFunction.apply(qk, x, rotations, side, heads)
    return rotary_formula(qk, x, rotations, side, heads, elu_plus_one)


def turn_formula(q, k, weight, rotations):
    b, heads, n, d = q.shape
    k = k * weight
    grid = (b, heads, *rotations.shape[:-2], d)
    return (k, *(rotate(t.reshape(grid), rotations).reshape(t.shape).to(q.dtype) for t in (q, k)))


class TurnedHeadsFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, weight, rotations):
        ctx.save_for_backward(q, k, weight, rotations)
        return _hip.turn_fwd(q, k, weight, rotations)

    @staticmethod
    def backward(ctx, *grads):
        inputs = ctx.saved_tensors
        return gradient_of(lambda *g: (*_hip.turn_bwd(*inputs[1:], *g), None),
                           lambda *g: differentiable_gradients(turn_formula, inputs, g), *grads)


def turned_heads(q, k, weight, rotations):
    """q, k [B, heads, N, d], weight [B, heads, N, 1], rotations [H, W, d / 2, 2] over the N tokens.  Returns (k * weight, q
    turned, k * weight turned)."""
    N, d = q.shape[-2:]
    pieces = d * q.element_size() // 16
    if (_takes(1, d, 1, q, k, weight) and pieces <= 64 and pieces & (pieces - 1) == 0 and type(rotations) is torch.Tensor and
            rotations.dtype == torch.float32 and rotations.device == q.device and not rotations.requires_grad and
            q.ndim == 4 and rotations.ndim == 4 and rotations.shape[0] * rotations.shape[1] == N and rotations.shape[2:] == (d // 2, 2) and
            k.shape == q.shape and weight.shape == (*q.shape[:-1], 1)):
        return TurnedHeadsFunction.apply(q, k, weight, rotations)
    return turn_formula(q, k, weight, rotations)


def merge_formula(o, o2, local, gate):
    out = merge_heads(o if o2 is None else torch.cat((o, o2), dim=-1)) + local
    return (out if gate is None else out * gate,)


class MergeHeadsFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, o, o2, local, gate):
        ctx.heads, ctx.halves = o.shape[1], o2 is not None
        ctx.save_for_backward(*((o, o2, local, gate) if gate is not None else (None,) * 4))
        return _hip.merge_fwd(o, o2, local, gate)

    @staticmethod
    def backward(ctx, g):
        inputs = ctx.saved_tensors  # o, o2, local, gate, or nothing without a gate

        def composed(g):
            if inputs[3] is not None:
                return differentiable_gradients(merge_formula, inputs, (g,))
            do = split_heads(g, ctx.heads)
            return (*(do.chunk(2, dim=-1) if ctx.halves else (do, None)), g, None)
        return gradient_of(lambda g: _hip.merge_bwd(g, ctx.heads, ctx.halves, *inputs), composed, g)


def merge_heads_with(o, o2, local, gate=None):
    """(heads + local) * gate as rows [B, N, C]: o [B, heads, N, d], or the halves o, o2 [B, heads, N, d / 2] of each head;
    local [B, N, C]; gate [B, N, C] or None."""
    heads, C, halves = o.shape[1], local.shape[-1], 1 if o2 is None else 2
    if (_takes(heads, C, halves, o, o2, local, gate) and local.shape == (o.shape[0], o.shape[2], heads * o.shape[3] * halves) and
            (o2 is None or o2.shape == o.shape) and (gate is None or gate.shape == local.shape)):
        return MergeHeadsFunction.apply(o, o2, local, gate)
    return merge_formula(o, o2, local, gate)[0]


def interpolate_formula(rows, tokens):
    return (F.interpolate(rows.transpose(1, 2), size=tokens, mode='linear').transpose(1, 2),)


class InterpolateTokensFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, rows, tokens):
        ctx.n = rows.shape[1]
        return _hip.interpolate_fwd(rows, tokens)

    @staticmethod
    def backward(ctx, g):
        def composed(g):  # linear in the rows: the gradient is that of any rows
            rows = torch.zeros(g.shape[0], ctx.n, g.shape[2], dtype=g.dtype, device=g.device, requires_grad=True)
            return differentiable_gradients(interpolate_formula, (rows, g.shape[1]), (g,))
        return gradient_of(lambda g: (_hip.interpolate_bwd(g, ctx.n), None), composed, g)


def interpolate_tokens(rows, tokens):
    """Token rows [B, n, C] linearly interpolated to [B, tokens, C] (corners not aligned)."""
    if (_takes(1, rows.shape[-1], 1, rows) and rows.ndim == 3 and tokens > 0 and rows.shape[1] * tokens < 1 << 28 and
            rows.shape[0] * tokens * rows.shape[2] < 1 << 31):
        return InterpolateTokensFunction.apply(rows, tokens)
    return interpolate_formula(rows, tokens)[0]
