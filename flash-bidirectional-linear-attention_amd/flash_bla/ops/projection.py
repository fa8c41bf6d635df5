"""Projections of token rows (nn.Linear) with the weight gradient on this package's kernel.

The blocks' projections contract 1e4 to 1e5 tokens into a weight gradient of a few hundred on a side, a shape for which
the library's GEMM fills a dozen CUs; `_hip.linear_wgrad` splits the tokens and takes the bias's gradient along.  The
forward and the input's gradient of a projection by itself stay plain library GEMMs (blocks that run whole: `_hip.mlla_fwd` and
the like, 16-bit types, on `csrc/fbla_gemm.hip`).
"""
import torch
import torch.nn as nn
import torch.nn.functional as F
from torch._C._functorch import is_legacy_batchedtensor as _is_batched  # what is_grads_batched makes of gradients
from torch.autograd import forward_ad

from flash_bla import _hip
from flash_bla.ops._check import untouched


class TokenLinearFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x, weight)
        ctx.with_bias = bias is not None
        return F.linear(x, weight, bias)

    @staticmethod
    def backward(ctx, g):
        x, weight = ctx.saved_tensors
        dx = g @ weight if ctx.needs_input_grad[0] else None
        with_bias = ctx.with_bias and ctx.needs_input_grad[2]

        def composed(g):
            rows = g.reshape(-1, g.shape[-1])
            return rows.t() @ x.reshape(-1, x.shape[-1]), rows.sum(0) if with_bias else None
        return (dx, *gradient_of(lambda g: _hip.linear_wgrad(g, x, with_bias), composed, g))


def eager_call():
    """Whether nothing traces, maps, watches or carries a tangent through torch's own operators here."""
    return not (torch.compiler.is_compiling() or torch._C._is_tracing() or forward_ad._current_level >= 0 or
                torch._C._are_functorch_transforms_active() or torch._C._len_torch_dispatch_stack())


def plain_tensors(*tensors):
    """Whether these are ordinary tensors in an ordinary eager call that casts nothing."""
    for t in tensors:
        if t is not None and type(t) is not torch.Tensor and type(t) is not nn.Parameter:
            return False
    return not torch.is_autocast_enabled() and eager_call()


def gradient_of(kernel, composition, *grads):
    """kernel(*grads), or composition(*grads) by torch's operators where the gradient is to be differentiated again, carries
    a tangent or is traced, and where the kernel cannot read the gradients: batches of gradients (is_grads_batched) and
    other tensors without memory of their own, whose address the kernel's binding asks for before it launches anything."""
    if torch.is_grad_enabled() or not eager_call():
        return composition(*grads)
    try:
        return kernel(*grads)
    except RuntimeError:
        if all(type(g) is torch.Tensor and not _is_batched(g) for g in grads):
            raise
    return composition(*grads)


def splits_tokens(tokens, M, N, with_bias, fp32):
    """Whether the kernel beats the library's gradient of an M x N weight (and its column sums for the bias).  Results with
    many tiles fill the GPU by themselves.  Measured, library + bias sum against the kernel, us:
    bf16: 1280 x 1280 over 1024 / 4096 tokens 22 + 13 / 26, 37 + 22 / 40; 1024 x 1024 over 2048 21 + 13 / 24; 640 x 640 over
    4096 29 + 19 / 21; 512 x 512 over 512 21 + 9 / 17.
    fp32: 512 x 256 over 50176 558 + 32 / 136; 320 x 320 over 8192 50 + 17 / 46; 640 x 640 over 4096 38 + 18 / 51; 1024 x 256
    over 3136 25 + 17 / 32; 1024 x 1024 over 2048 39 + 13 / 55; 256 x 128 over 1024 22 + 11 / 28."""
    if fp32:
        return M * N <= 1 << 19 if with_bias else M * N <= 1 << 17 and tokens >= 8192
    return M * N <= (1 << 21 if with_bias else 1 << 19)


def runs_on_rows(x, weight, bias):
    """Whether the weight gradient of F.linear(x, weight, bias) is left to the kernel."""
    if not (weight.requires_grad and x.is_cuda and torch.is_grad_enabled() and x.ndim >= 2 and x.numel() > 0 and
            x.dtype in (torch.float16, torch.bfloat16, torch.float32) and x.shape[-1] == weight.shape[1]):
        return False
    (M, N), piece, tokens = weight.shape, 16 // x.element_size(), x.numel() // x.shape[-1]
    return (weight.dtype == x.dtype and weight.device == x.device and (bias is None or bias.dtype == x.dtype) and
            M % piece == 0 and N % piece == 0 and tokens <= 1 << 30 and
            splits_tokens(tokens, M, N, bias is not None, x.dtype == torch.float32) and plain_tensors(x, weight, bias))


def token_linear(x, weight, bias):
    """F.linear whose backward takes the weight and bias gradients from the token-splitting kernel where that is the
    faster of the two."""
    if runs_on_rows(x, weight, bias):
        return TokenLinearFunction.apply(x, weight, bias)
    return F.linear(x, weight, bias)


def trains(x):
    """Whether a call on x can need the gradients at all: a tensor (no proxy of one), grad mode, no trace."""
    return type(x) is torch.Tensor and torch.is_grad_enabled() and not torch._C._is_tracing()


def project(module, x):
    """module(x), a plain nn.Linear as token_linear.  The blocks hold plain nn.Linear modules and call them through this:
    what replaces, wraps, traces or looks for modules by their type finds them as they always were."""
    if trains(x) and untouched(module, nn.Linear):
        weight, bias = module.weight, module.bias
        if runs_on_rows(x, weight, bias):
            return TokenLinearFunction.apply(x, weight, bias)
    return module(x)


class TokenLinear(nn.Linear):
    """token_linear as a module of its own."""

    def forward(self, x):
        return token_linear(x, self.weight, self.bias)
