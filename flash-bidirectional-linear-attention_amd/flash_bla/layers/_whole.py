"""Blocks as one native call a direction (csrc/fbla_torch.cpp).

Issued step by step from Python, a block's training step on few tokens is bound by the host: every projection, feature map,
operator and merge is a node of the autograd graph with its checks, its Python calls and its bookkeeping.  Where nothing
looks between the steps - an ordinary eager call of the block's own class on plain modules, without hooks, of the shapes that
all its fused steps take - the block is one node instead.  Its forward and backward do what the steps do, 16-bit types on kernels
that only whole blocks have: projections with residuals and second products in their sums, the norm and activation between them
(csrc/fbla_gemm.hip), and with heads of 32 channels PolaFormer's and MLLA's attention on the projections' rows (csrc/fbla_rows.hip).
Everything else (autocast among it) runs step by step (`_steps` of the block), and so does a gradient that is to be differentiated
again or that the kernels cannot read: it is composed by running the steps on what the node saved.

Host time of a forward / a training step, steps from Python through ctypes and here, us, in the slower of the host's two states
(the faster one takes two thirds): mlla 107 / 450 -> 31 / 175, pola 198 / 800 -> 44 / 275, with spatial reduction 348 / 1280 -> 114 /
590, focused 161 / 680 -> 57 / 310 (2 x 14x14 x 64 bf16), linfusion 249 / 1100 -> 74 / 500 (1 x 16x16 x 320 fp16).  What is left is the
engine's hand-over to its thread (a node of the graph that does nothing costs 33 or 63 us there), torch's own modules and GEMM calls
(17 us each, a launch of this package 4), and the launches.
"""
import contextlib

import torch
import torch.nn as nn
from torch._C import _functorch
from torch.nn.modules.module import _has_any_global_hook
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from flash_bla import _hip
from flash_bla.ops.projection import eager_call, gradient_of, splits_tokens


def _bare(kind, **members):
    """A module of the class that holds these and nothing else: what `_steps` of a block and `project` look at."""
    module = kind.__new__(kind)
    nn.Module.__init__(module)
    for name, value in members.items():
        setattr(module, name, value)
    return module


def _linear(weight, bias):
    return _bare(nn.Linear, weight=weight, bias=bias)


def _convolution(weight, bias):
    """As _same_convolution knows it."""
    Cw, _, K, _ = weight.shape
    return _bare(nn.Conv2d, weight=weight, bias=bias, in_channels=Cw, out_channels=Cw, groups=Cw, kernel_size=(K, K), stride=(1, 1),
                 padding=(K // 2, K // 2), dilation=(1, 1), padding_mode='zeros')


def _batch_of(g):
    """A batch of gradients (is_grads_batched, torch.func.vmap) as an ordinary tensor with the batch first, what wraps results
    like it, and a context in which ordinary tensors are no more than that; None for any other gradient."""
    if _functorch.is_legacy_batchedtensor(g):
        values = torch._remove_batch_dim(g, 1, 1, 0)  # (batched at another level, it stays a batch)
        if not _functorch.is_legacy_batchedtensor(values):
            return values, lambda t: torch._add_batch_dim(t, 0, 1), contextlib.nullcontext
    elif _functorch.is_batchedtensor(g):
        level, values = _functorch.maybe_get_level(g), _functorch.get_unwrapped(g).movedim(_functorch.maybe_get_bdim(g), 0)
        if not _functorch.is_functorch_wrapped_tensor(values):
            from torch._functorch.pyfunctorch import temporarily_clear_interpreter_stack  # (a private name: needed here only)
            return values, lambda t: _functorch._add_batch_dim(t, 0, level), temporarily_clear_interpreter_stack
    return None


class WholeBlockFunction(torch.autograd.Function):
    """call: the block's native pair and the same as `_steps` of a block that holds the inputs (below), with the module's numbers
    as they are when it is called: by the time of the backward a schedule may have moved them, or hooks and other parameters
    taken their place.  inputs: the block's rows and parameters, some of them None, and what else the backward reads."""

    @staticmethod
    def forward(ctx, call, *inputs):
        ctx.call = call
        out, *saved = call.run(inputs)
        ctx.save_for_backward(*inputs, *saved)
        return out

    @staticmethod
    def backward(ctx, g):
        call, tensors = ctx.call, ctx.saved_tensors
        need = ctx.needs_input_grad[1:]
        inputs, saved = tensors[:len(need)], tensors[len(need):]

        def composed(g):
            batch = None if torch.is_grad_enabled() else _batch_of(g)
            if batch is not None:  # (the node has to give all its gradients, and the operators' kernels take one at a time)
                values, wrapped, ordinary = batch
                with ordinary():
                    each = [call.run_backward(e, inputs, saved, need) for e in values.unbind()]
                    stacked = [None if t[0] is None else torch.stack(t) for t in zip(*each)]
                return [None if t is None else wrapped(t) for t in stacked]
            with torch.enable_grad():  # (through aliases: the inputs may depend on one another, or be one tensor)
                aliases = [t.view_as(t) if t is not None and t.requires_grad else t for t in inputs]
                out = call.steps(*aliases)
            wanted = [a for a, wants in zip(aliases, need) if wants]
            got = iter(torch.autograd.grad(out, wanted, g, create_graph=torch.is_grad_enabled(), allow_unused=True))
            return [next(got) if wants else None for wants in need]
        return (None, *gradient_of(lambda g: call.run_backward(g, inputs, saved, need), composed, g))


def _run(call, inputs):
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in inputs):
        return WholeBlockFunction.apply(call, *inputs)
    return call.run(inputs, trains=False)[0]


def _watched():
    """Whether a torch function mode would see, or replace, the operators that the steps call (a default device is one, too, and
    neither)."""
    return torch._C._len_torch_function_stack() and any(type(mode) is not DeviceContext for mode in _get_current_function_mode_stack())


def _ordinary(block, kind, x, modules):
    """An eager call of the block's own class on GPU rows, nothing around or in place of its modules' forwards."""
    return (type(x) is torch.Tensor and x.is_cuda and x.ndim == 3 and type(block) is kind and not torch.is_autocast_enabled() and
            eager_call() and not _watched() and not _has_any_global_hook() and _hip.untouched_modules(modules))


def _same_convolution(conv):
    """Stride 1 and "same" zero padding for the filters that it holds; their shape is compared natively."""
    Cw, K = conv.weight.shape[0], conv.weight.shape[-1]
    return (conv.kernel_size == (K, K) and conv.padding == (K // 2, K // 2) and conv.padding_mode == 'zeros' and
            conv.stride == (1, 1) and conv.dilation == (1, 1) and conv.groups == Cw)


def _splits(rows, weight, bias):
    """Whether a projection's weight gradient is the token-splitting kernel's."""
    return splits_tokens(rows.numel() // rows.shape[-1], *weight.shape, bias is not None, rows.dtype == torch.float32)


class _Mlla:
    """inputs: x, parameters, rotations."""

    def __init__(self, block, kind, rope, side):
        self.kind, self.rope, self.side, self.heads = kind, rope, side, block.num_heads

    def steps(self, x, w, b, conv_w, conv_b, rotations):
        return _bare(self.kind, num_heads=self.heads, qk=_linear(w, b), lepe=_convolution(conv_w, conv_b),
                     rope=_bare(self.rope, rotations=rotations))._steps(x, True)

    def run(self, inputs, trains=True):
        *inputs, rotations = inputs
        return _hip.mlla_fwd(inputs[0], inputs[1:], rotations, self.side, self.heads, trains)

    def run_backward(self, g, inputs, saved, need):
        x, w, b, conv_w, _, rotations = inputs
        return [*_hip.mlla_bwd(g, x, w, conv_w, rotations, saved, self.side, self.heads, need[:5], _splits(x, w, b)), None]


def mlla(block, kind, rope, x):
    """The block's output, or None where it is not to run whole."""
    if not _ordinary(block, kind, x, [(block.qk, nn.Linear), (block.lepe, nn.Conv2d), (block.rope, rope)]):
        return None
    side, rotations = int(x.shape[1] ** 0.5), block.rope.rotations
    params = (block.qk.weight, block.qk.bias, block.lepe.weight, block.lepe.bias)
    if not (type(rotations) is torch.Tensor and _hip.plain_gpu_tensors(x, *params) and _same_convolution(block.lepe) and
            _hip.mlla_fits(x, params, rotations, side, block.num_heads)):
        return None
    return _run(_Mlla(block, kind, rope, side), (x, *params, rotations))


class _Pvt:
    """PolaFormer's and FLatten's blocks.  inputs: x, the rows of keys and values (None: x), parameters."""

    def __init__(self, block, kind, H, W):
        self.kind, self.H, self.W, self.heads, self.sr_ratio = kind, H, W, block.num_heads, block.sr_ratio

    def _block(self, kv_w, kv_b, pe, scale, conv_w, conv_b, proj_w, proj_b, **more):
        return _bare(self.kind, num_heads=self.heads, sr_ratio=self.sr_ratio, kv=_linear(kv_w, kv_b), positional_encoding=pe,
                     scale=scale, dwc=_convolution(conv_w, conv_b), proj=_linear(proj_w, proj_b), **more)

    def _split(self, inputs, saved):
        x, src, *p = inputs
        q_w, q_b, kv_w, kv_b = p[:4]
        return _splits(x, q_w, q_b), _splits(x if src is None else src, kv_w, kv_b), _splits(x, p[-2], p[-1])


class _Pola(_Pvt):
    def __init__(self, block, kind, H, W):
        super().__init__(block, kind, H, W)
        self.alpha = block.alpha

    def steps(self, x, src, q_w, q_b, kv_w, kv_b, pe, scale, power, *more):
        block = self._block(kv_w, kv_b, pe, scale, *more, qg=_linear(q_w, q_b), power=power, alpha=self.alpha)
        return block._steps(x, src, self.H, self.W, True)

    def run(self, inputs, trains=True):
        x, src, *p = inputs
        return _hip.pola_fwd(x, x if src is None else src, p, self.alpha, self.H, self.W, self.heads, trains)

    def run_backward(self, g, inputs, saved, need):
        x, src, *p = inputs
        return _hip.pola_bwd(g, x, x if src is None else src, src is None, p, saved, self.alpha, self.H, self.W,
                             self.heads, need, self._split(inputs, saved))


class _Focused(_Pvt):
    def steps(self, x, src, q_w, q_b, *more):
        return self._block(*more, q=_linear(q_w, q_b), focusing_factor=3)._steps(x, src, self.H, self.W, True)

    def run(self, inputs, trains=True):
        x, src, *p = inputs
        return _hip.focused_fwd(x, x if src is None else src, p, self.H, self.W, self.heads, trains)

    def run_backward(self, g, inputs, saved, need):
        x, src, *p = inputs
        return _hip.focused_bwd(g, x, x if src is None else src, src is None, p, saved, self.H, self.W, self.heads, need,
                                self._split(inputs, saved))


def _pvt(call, block, fits, params, x, src):
    H, W = call.H, call.W
    if not (type(H) is int and type(W) is int and (src is None or type(src) is torch.Tensor) and
            _hip.plain_gpu_tensors(x, src, *params) and _same_convolution(block.dwc) and
            fits(x, x if src is None else src, params, H, W, call.heads)):
        return None
    return _run(call, (x, src, *params))


def pola(block, kind, x, src, H, W):
    if not (type(block.alpha) in (int, float) and block.alpha >= 0 and _ordinary(block, kind, x, [
            (block.qg, nn.Linear), (block.kv, nn.Linear), (block.proj, nn.Linear), (block.dwc, nn.Conv2d)])):
        return None
    return _pvt(_Pola(block, kind, H, W), block, _hip.pola_fits, (
        block.qg.weight, block.qg.bias, block.kv.weight, block.kv.bias, block.positional_encoding, block.scale, block.power,
        block.dwc.weight, block.dwc.bias, block.proj.weight, block.proj.bias), x, src)


def focused(block, kind, x, src, H, W):
    factor = block.focusing_factor
    if not (type(factor) in (int, float) and factor == 3 and _ordinary(block, kind, x, [
            (block.q, nn.Linear), (block.kv, nn.Linear), (block.proj, nn.Linear), (block.dwc, nn.Conv2d)])):
        return None
    return _pvt(_Focused(block, kind, H, W), block, _hip.focused_fits, (
        block.q.weight, block.q.bias, block.kv.weight, block.kv.bias, block.positional_encoding, block.scale, block.dwc.weight,
        block.dwc.bias, block.proj.weight, block.proj.bias), x, src)


class _LinFusion:
    """inputs: x, parameters (both paths' first projection, norm and second projection, then queries, keys, values, output), the
    packed batch's offsets."""

    def __init__(self, block, kind):
        paths = block.to_q_, block.to_k_
        self.kind, self.heads = kind, block.heads
        self.eps, self.slope = tuple(p[1].eps for p in paths), tuple(p[2].negative_slope for p in paths)

    def steps(self, x, *p):
        def path(i):
            in_w, in_b, norm_w, norm_b, out_w, out_b = p[6 * i:6 * i + 6]
            norm = _bare(nn.LayerNorm, normalized_shape=in_w.shape[:1], weight=norm_w, bias=norm_b, eps=self.eps[i])
            return nn.Sequential(_linear(in_w, in_b), norm, nn.LeakyReLU(self.slope[i]), _linear(out_w, out_b))
        q, k, v, out = (_linear(*p[i:i + 2]) for i in range(12, 20, 2))
        return _bare(self.kind, heads=self.heads, to_q_=path(0), to_k_=path(1), to_q=q, to_k=k, to_v=v, to_out=[out])._steps(x)

    def run(self, inputs, trains=True):
        x, *p, cu = inputs
        return _hip.linfusion_fwd(x, cu, p, self.eps, self.slope, self.heads, trains)

    def run_backward(self, g, inputs, saved, need):
        x, *p, cu = inputs
        split = [_splits(x, p[i], p[i + 1]) for i in (0, 4, 6, 10, 12, 14, 16, 18)]
        return [*_hip.linfusion_bwd(g, x, cu, p, saved, self.slope, need[:-1], split), None]


def _keeps_signs(activation):
    """Whether LeakyReLU's output has its input's sign, from which the backward takes the activation's gradient."""
    return type(activation.negative_slope) in (int, float) and activation.negative_slope >= 0


def linfusion(block, kind, x, cu):
    """cu(): the packed batch's offsets."""
    paths = (block.to_q_, block.to_k_)
    if type(x) is not torch.Tensor or not x.is_cuda or not all(type(p) is nn.Sequential and len(p) == 4 for p in paths):
        return None
    projections = (block.to_q, block.to_k, block.to_v, block.to_out[0])
    kinds = (nn.Linear, nn.LayerNorm, nn.LeakyReLU, nn.Linear)
    if not _ordinary(block, kind, x, [(p, nn.Sequential) for p in paths] + [m for p in paths for m in zip(p, kinds)] +
                     [(m, nn.Linear) for m in projections]):
        return None
    params = [t for p in paths for i in (0, 1, 3) for t in (p[i].weight, p[i].bias)]
    params += [t for m in projections for t in (m.weight, m.bias)]
    if not (all(_keeps_signs(p[2]) for p in paths) and _hip.plain_gpu_tensors(x, *params) and
            all(tuple(p[1].normalized_shape) == tuple(p[0].weight.shape[:1]) for p in paths) and
            _hip.linfusion_fits(x, params, block.heads)):
        return None
    return _run(_LinFusion(block, kind), (x, *params, cu()))
